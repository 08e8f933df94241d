// The few runtime calls csrc/host_copy.hip makes, on the host: device memory is host
// memory, a stream finishes its earlier work `busy` seconds after the first wait for
// it, an event is recorded only on a stream of its own device.
#pragma once
#include <chrono>
#include <cstddef>
#include <cstdlib>
#include <cstring>
#include <thread>

enum hipError_t { hipSuccess = 0, hipErrorInvalidValue = 1, hipErrorInvalidHandle = 400, hipErrorUnknown = 999 };
enum hipMemcpyKind { hipMemcpyHostToDevice, hipMemcpyDeviceToHost };
enum hipMemoryType { hipMemoryTypeUnregistered, hipMemoryTypeHost };
struct hipPointerAttribute_t {
    hipMemoryType type;
};
struct FakeStream {
    int device = 0;
    double busy = 0.0;
};
struct FakeEvent {
    int device = 0;
};
using hipStream_t = FakeStream*;
using hipEvent_t = FakeEvent*;
constexpr unsigned hipHostMallocDefault = 0, hipEventDisableTiming = 2;

namespace fake {
inline int current = 0;     // device
inline int live = 0;        // events and buffers not yet freed
inline int copies = 0;      // asynchronous copies so far
inline int fail_at = -1;    // the copy that fails
inline int pinned = 0;      // pinned allocations so far
inline void wait(FakeStream* s)
{
    if (s->busy > 0.0) std::this_thread::sleep_for(std::chrono::duration<double>(s->busy));
    s->busy = 0.0;
}
}  // namespace fake

inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipGetDevice(int* d) { return *d = fake::current, hipSuccess; }
inline hipError_t hipSetDevice(int d) { return fake::current = d, hipSuccess; }
inline hipError_t hipStreamGetDevice(hipStream_t s, int* d) { return *d = s->device, hipSuccess; }
inline hipError_t hipPointerGetAttributes(hipPointerAttribute_t*, const void*) { return hipErrorInvalidValue; }
inline hipError_t hipHostMalloc(void** p, size_t n, unsigned)
{
    *p = std::malloc(n);
    fake::live++;
    fake::pinned++;
    return hipSuccess;
}
inline hipError_t hipHostFree(void* p)
{
    std::free(p);
    fake::live--;
    return hipSuccess;
}
inline hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned)
{
    *e = new FakeEvent{fake::current};
    fake::live++;
    return hipSuccess;
}
inline hipError_t hipEventDestroy(hipEvent_t e)
{
    delete e;
    fake::live--;
    return hipSuccess;
}
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t s)
{
    return e->device == s->device ? hipSuccess : hipErrorInvalidHandle;
}
inline hipStream_t& fake_last_stream()
{
    static hipStream_t s = nullptr;
    return s;
}
inline hipError_t hipMemcpyAsync(void* dst, const void* src, size_t n, hipMemcpyKind, hipStream_t s)
{
    if (fake::copies++ == fake::fail_at) return hipErrorUnknown;
    std::memcpy(dst, src, n);
    fake_last_stream() = s;
    return hipSuccess;
}
inline hipError_t hipEventSynchronize(hipEvent_t)
{
    fake::wait(fake_last_stream());
    return hipSuccess;
}
inline hipError_t hipStreamSynchronize(hipStream_t s)
{
    fake::wait(s);
    return hipSuccess;
}
