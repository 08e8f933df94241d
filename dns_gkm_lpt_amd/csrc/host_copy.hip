// host_copy.hip -- see host_copy.hpp.
//
// What bounds a large copy to or from pageable memory is the host: one thread
// faulting in the caller's fresh pages and moving the bytes.  Here the device
// copies chunks into a ring of pinned buffers while up to eight threads move
// earlier chunks on, each a slice of every chunk.  A 512^3 state (5.6 GB) comes
// down in 117 ms (47 GB/s) instead of 561 and goes up in 111 instead of 199; a
// 128^3 one (96 MB) 2.7-4.5 instead of 9.8 and 2.3 instead of 3.6.  Slices of
// 1 MB: with 256 KB several threads fault in the same 2 MB page (27 GB/s at
// 256^3 against 46); 14 threads are no faster.  Below 32 MB the plain copy is
// used: at 14 MB (64^3) it takes 0.86 ms down against 1.2, and the buffers' own
// allocation (about 1.5 ms) would not come back in a short-lived context.
#include "host_copy.hpp"

#include <sched.h>

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstdio>
#include <cstring>
#include <mutex>
#include <thread>
#include <vector>

namespace gkm {

namespace {

constexpr size_t kSlice = size_t(1) << 20;

// CPUs the process may use: its affinity, and a container's CPU quota, under which
// more threads than it pays for only stop each other
int usable_cpus()
{
    cpu_set_t set;
    CPU_ZERO(&set);
    int n = sched_getaffinity(0, sizeof(set), &set) == 0 ? CPU_COUNT(&set) : 1;
    double quota = 0.0, period = 0.0;
    if (FILE* f = std::fopen("/sys/fs/cgroup/cpu.max", "r")) {  // "max <period>" without a limit
        if (std::fscanf(f, "%lf %lf", &quota, &period) == 2 && period > 0.0) n = std::min(n, (int)(quota / period));
        std::fclose(f);
    }
    return std::max(1, n);
}

// the device of a stream made current, and the caller's again afterwards
class OnDeviceOf {
  public:
    explicit OnDeviceOf(hipStream_t s)
    {
        int dev = -1;
        ok_ = hipGetDevice(&was_) == hipSuccess && hipStreamGetDevice(s, &dev) == hipSuccess;
        if (ok_ && dev != was_) {
            ok_ = hipSetDevice(dev) == hipSuccess;
            changed_ = ok_;
        }
        if (!ok_) (void)hipGetLastError();
    }
    ~OnDeviceOf()
    {
        if (changed_) (void)hipSetDevice(was_);
    }
    bool ok() const { return ok_; }

  private:
    int was_ = 0;
    bool ok_ = false, changed_ = false;
};

// memory the runtime knows (pinned, managed, on a device): the device reaches it
// itself, and host code may not
bool known_to_runtime(const void* p)
{
    hipPointerAttribute_t a{};
    if (hipPointerGetAttributes(&a, p) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    return a.type != hipMemoryTypeUnregistered;
}

struct Chunk {
    char *host, *dev;
    size_t bytes;
};

}  // namespace

void HostPipe::release()
{
    for (hipEvent_t& e : ev_) {
        if (e) (void)hipEventDestroy(e);
        e = nullptr;
    }
    if (buf_) (void)hipHostFree(buf_);
    buf_ = nullptr;
    chunk_ = 0;
}

// pinned buffers for copies of `bytes` in all on s's device, whichever is current
// (an event is recorded on its own device's streams only); false if there are none
// to be had
bool HostPipe::ready(size_t bytes, hipStream_t s)
{
    const size_t want = std::min(kChunk, ((bytes + kDepth - 1) / kDepth + kSlice - 1) / kSlice * kSlice);
    if (chunk_ >= want) return true;
    release();
    const OnDeviceOf here(s);
    if (!here.ok()) return false;
    if (hipHostMalloc(reinterpret_cast<void**>(&buf_), kDepth * want, hipHostMallocDefault) != hipSuccess) {
        (void)hipGetLastError();
        buf_ = nullptr;
        return false;
    }
    for (hipEvent_t& e : ev_)
        if (hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) {
            (void)hipGetLastError();
            e = nullptr;
            release();
            return false;
        }
    chunk_ = want;
    return true;
}

hipError_t HostPipe::plain(const CopySeg* seg, int n, hipStream_t s, bool to_host)
{
    for (int i = 0; i < n; i++) {
        const hipError_t e = to_host ? hipMemcpyAsync(seg[i].host, seg[i].dev, seg[i].bytes, hipMemcpyDeviceToHost, s)
                                     : hipMemcpyAsync(seg[i].dev, seg[i].host, seg[i].bytes, hipMemcpyHostToDevice, s);
        if (e != hipSuccess) return e;
    }
    return to_host ? hipStreamSynchronize(s) : hipSuccess;
}

hipError_t HostPipe::run(const CopySeg* seg, int n, hipStream_t s, bool to_host)
{
    size_t total = 0;
    for (int i = 0; i < n; i++) total += seg[i].bytes;
    if (total < kPipeMin) return plain(seg, n, s, to_host);
    for (int i = 0; i < n; i++)
        if (known_to_runtime(seg[i].host)) return plain(seg, n, s, to_host);
    const int nthr = (int)std::min<size_t>(std::min(usable_cpus(), 8), total / (size_t(2) << 20) + 1);
    if (nthr < 2 || !ready(total, s)) return plain(seg, n, s, to_host);
    // The threads' waits spin, which is for the times between two chunks only: while
    // the stream's earlier work runs, they sleep (down: until the first chunk has
    // arrived) or are not there yet (up).
    if (!to_host) {
        const hipError_t before = hipStreamSynchronize(s);
        if (before != hipSuccess) return before;
    }
    std::mutex gate_mutex;
    std::condition_variable gate;

    std::vector<Chunk> chunks;
    std::vector<std::thread> threads;
    std::atomic<int> next{0}, filled{0};  // slices handed out; chunks the copying threads may start on
    std::atomic<bool> stop{false};
    std::atomic<int> left[kDepth];        // slices of the buffer's chunk not yet moved
    for (auto& l : left) l.store(0, std::memory_order_relaxed);
    try {
        for (int i = 0; i < n; i++)
            for (size_t o = 0; o < seg[i].bytes; o += chunk_)
                chunks.push_back({static_cast<char*>(seg[i].host) + o, static_cast<char*>(seg[i].dev) + o,
                                  std::min(chunk_, seg[i].bytes - o)});
        threads.reserve(nthr);
    } catch (...) {
        return plain(seg, n, s, to_host);
    }
    const int nch = (int)chunks.size(), per = (int)(chunk_ / kSlice);
    // one slice of a chunk between its buffer and the caller's memory
    auto move = [&](int k) {
        const int i = k / per;
        const size_t o = (size_t)(k % per) * kSlice;
        if (o < chunks[i].bytes) {
            char* pinned = buf_ + (size_t)(i % kDepth) * chunk_ + o;
            const size_t b = std::min(kSlice, chunks[i].bytes - o);
            if (to_host) std::memcpy(chunks[i].host + o, pinned, b);
            else std::memcpy(pinned, chunks[i].host + o, b);
        }
        left[i % kDepth].fetch_sub(1, std::memory_order_release);
    };
    auto worker = [&] {
        {
            std::unique_lock<std::mutex> hold(gate_mutex);
            gate.wait(hold, [&] { return filled.load(std::memory_order_relaxed) > 0 || stop.load(std::memory_order_relaxed); });
        }
        for (;;) {
            const int k = next.fetch_add(1, std::memory_order_relaxed);
            if (k >= nch * per) return;
            while (filled.load(std::memory_order_acquire) <= k / per) {
                if (stop.load(std::memory_order_relaxed)) return;
                std::this_thread::yield();
            }
            move(k);
        }
    };
    for (int t = 0; t < nthr; t++) {
        try {
            threads.emplace_back(worker);
        } catch (...) {
            break;  // fewer threads
        }
    }
    if (threads.empty()) return plain(seg, n, s, to_host);

    auto open_gate = [&] {
        { std::lock_guard<std::mutex> hold(gate_mutex); }
        gate.notify_all();
    };
    // buffer b's last chunk moved on by the threads
    auto drained = [&](int b) {
        while (left[b].load(std::memory_order_acquire) > 0) std::this_thread::yield();
    };
    hipError_t e = hipSuccess;
    if (to_host) {
        int sent = 0;
        for (int i = 0; i < nch && e == hipSuccess; i++) {
            for (; sent < nch && sent < i + kDepth && e == hipSuccess; sent++) {
                const int b = sent % kDepth;
                if (sent > i && left[b].load(std::memory_order_acquire) > 0) break;  // still being moved: come back
                drained(b);
                e = hipMemcpyAsync(buf_ + (size_t)b * chunk_, chunks[sent].dev, chunks[sent].bytes, hipMemcpyDeviceToHost, s);
                if (e == hipSuccess) e = hipEventRecord(ev_[b], s);
            }
            if (e == hipSuccess) e = hipEventSynchronize(ev_[i % kDepth]);
            if (e == hipSuccess) {
                left[i % kDepth].store(per, std::memory_order_relaxed);
                filled.store(i + 1, std::memory_order_release);
                if (i == 0) open_gate();
            }
        }
    } else {
        // the threads fill a buffer once its previous chunk is on the device
        int open = 0;
        for (int i = 0; i < nch && e == hipSuccess; i++) {
            for (; open < nch && open < i + kDepth && e == hipSuccess; open++) {
                if (open >= kDepth) e = hipEventSynchronize(ev_[open % kDepth]);
                left[open % kDepth].store(per, std::memory_order_relaxed);
                filled.store(open + 1, std::memory_order_release);
                if (open == 0) open_gate();
            }
            if (e != hipSuccess) break;
            const int b = i % kDepth;
            drained(b);
            e = hipMemcpyAsync(chunks[i].dev, buf_ + (size_t)b * chunk_, chunks[i].bytes, hipMemcpyHostToDevice, s);
            if (e == hipSuccess) e = hipEventRecord(ev_[b], s);
        }
    }
    if (e != hipSuccess) stop.store(true, std::memory_order_relaxed);
    open_gate();
    for (auto& t : threads) t.join();
    const hipError_t es = hipStreamSynchronize(s);
    return e != hipSuccess ? e : es;
}

}  // namespace gkm
