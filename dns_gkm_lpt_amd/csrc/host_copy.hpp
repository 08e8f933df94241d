// host_copy.hpp -- copies between caller-owned (pageable) host memory and the
// device, through pinned buffers, with several host threads moving the data
// between the pinned buffers and the caller's.
#pragma once
#include <hip/hip_runtime.h>
#include <cstddef>

namespace gkm {

struct CopySeg {
    void* host;
    void* dev;
    size_t bytes;
};

// One pipe serves one thread and one stream at a time (a context's).  The pinned
// buffers (at most kDepth x kChunk bytes) are allocated by the first copy that
// uses them and freed by release().
class HostPipe {
  public:
    // the copies of n segments after the work on s.  to_host returns when the last
    // byte has arrived.  to_device may leave a small copy queued: whoever owns the
    // memory waits for s before its caller gets it back.
    hipError_t to_host(const CopySeg* seg, int n, hipStream_t s) { return run(seg, n, s, true); }
    hipError_t to_device(const CopySeg* seg, int n, hipStream_t s) { return run(seg, n, s, false); }
    void release();

    static constexpr size_t kPipeMin = size_t(32) << 20;  // smaller copies go straight
    static constexpr int kDepth = 4;
    static constexpr size_t kChunk = size_t(8) << 20;

  private:
    hipError_t run(const CopySeg* seg, int n, hipStream_t s, bool to_host);
    hipError_t plain(const CopySeg* seg, int n, hipStream_t s, bool to_host);
    bool ready(size_t bytes, hipStream_t s);

    char* buf_ = nullptr;
    size_t chunk_ = 0;  // bytes of each of the kDepth buffers
    hipEvent_t ev_[kDepth] = {};
};

}  // namespace gkm
