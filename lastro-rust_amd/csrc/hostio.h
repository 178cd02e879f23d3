// Small transfers between a handle's stream and the caller's memory through one pinned buffer of the handle. A copy
// to pageable memory waits for the stream and for its own round trip, one after the other; here the results of a call
// are registered, one kernel writes them all into the mapped buffer behind the call's work, and after the call's one
// wait they are copied to the caller. Inputs are copied into the buffer and read from there in stream order.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <cstring>

namespace moert {

struct HostSegs {
  static constexpr int kMax = 16;
  const void* src[kMax];
  unsigned off[kMax], words[kMax];  // place in the buffer (64-byte steps), 4-byte words
};

// grid (x, segments): segment blockIdx.y, 16 bytes a thread where its source allows
__global__ __launch_bounds__(256) static void k_host_gather(HostSegs s, uint8_t* __restrict__ out) {
  const int i = blockIdx.y;
  const unsigned n = s.words[i], t = blockIdx.x * 256 + threadIdx.x, step = gridDim.x * 256;
  const uint32_t* src = reinterpret_cast<const uint32_t*>(s.src[i]);
  uint32_t* dst = reinterpret_cast<uint32_t*>(out + s.off[i]);
  unsigned done = 0;
  if ((reinterpret_cast<uintptr_t>(src) & 15) == 0) {
    const uint4* s4 = reinterpret_cast<const uint4*>(src);
    uint4* d4 = reinterpret_cast<uint4*>(dst);
    for (unsigned j = t; j < n / 4; j += step) d4[j] = s4[j];
    done = n / 4 * 4;
  }
  for (unsigned j = done + t; j < n; j += step) dst[j] = src[j];
}

class HostIo {
 public:
  // a buffer of `bytes` (one handle's; the handle is used by one thread at a time)
  hipError_t create(size_t bytes) {
    hipError_t e = hipHostMalloc((void**)&buf_, bytes, hipHostMallocMapped);
    if (e != hipSuccess) return e;
    cap_ = bytes;
    return hipHostGetDevicePointer((void**)&dev_, buf_, 0);
  }
  ~HostIo() {
    if (buf_) (void)hipHostFree(buf_);
  }

  // dev[0, bytes) = src, in stream order; src is free on return
  hipError_t in(hipStream_t s, void* dev, const void* src, size_t bytes) {
    if (!src && bytes) return hipErrorInvalidValue;
    if (!fits(bytes)) return hipMemcpyAsync(dev, src, bytes, hipMemcpyHostToDevice, s);
    uint8_t* p = buf_ + used_;
    std::memcpy(p, src, bytes);
    take(bytes);
    return hipMemcpyAsync(dev, p, bytes, hipMemcpyHostToDevice, s);
  }
  // dst[0, bytes) = dev, as it stands behind the work queued so far; there after finish()
  hipError_t out(hipStream_t s, void* dst, const void* dev, size_t bytes) {
    if (!dst && bytes) return hipErrorInvalidValue;  // refused here: finish() would copy into it
    if (bytes % 4 || (reinterpret_cast<uintptr_t>(dev) & 3) || !fits(bytes) || n_outs_ == kOuts)
      return hipMemcpyAsync(dst, dev, bytes, hipMemcpyDeviceToHost, s);
    segs_.src[n_] = dev;
    segs_.off[n_] = (unsigned)used_;
    segs_.words[n_] = (unsigned)(bytes / 4);
    outs_[n_outs_++] = Out{dst, used_, bytes};
    take(bytes);
    return ++n_ == HostSegs::kMax ? flush(s) : hipSuccess;
  }
  // Queues the registered results; call before waiting for the stream.
  hipError_t flush(hipStream_t s) {
    if (!n_) return hipSuccess;
    unsigned most = 0;
    for (int i = 0; i < n_; i++) most = segs_.words[i] > most ? segs_.words[i] : most;
    const unsigned blocks = (most / 4 + 255) / 256;
    hipLaunchKernelGGL(k_host_gather, dim3(blocks < 1 ? 1 : blocks > 64 ? 64 : blocks, n_), 256, 0, s, segs_, dev_);
    n_ = 0;
    return hipGetLastError();
  }
  // After the stream is idle: results to the caller's memory (dropped without `ok`), the buffer free again.
  void finish(bool ok) {
    if (ok)
      for (int i = 0; i < n_outs_; i++) std::memcpy(outs_[i].dst, buf_ + outs_[i].off, outs_[i].bytes);
    n_outs_ = 0;
    used_ = 0;
    n_ = 0;
  }

  // Drops what a failed call left, once the stream no longer reads the buffer.
  hipError_t restart(hipStream_t s) {
    if (!used_) return hipSuccess;
    const hipError_t e = hipStreamSynchronize(s);
    finish(false);
    return e;
  }

 private:
  struct Out {
    void* dst;
    size_t off, bytes;
  };
  bool fits(size_t bytes) const { return used_ + bytes <= cap_; }
  void take(size_t bytes) { used_ = (used_ + bytes + 63) / 64 * 64; }
  uint8_t *buf_ = nullptr, *dev_ = nullptr;
  size_t cap_ = 0, used_ = 0;
  HostSegs segs_{};
  int n_ = 0;
  static constexpr int kOuts = 64;  // results of a call; a further one is a plain copy. Fixed: no call allocates
  Out outs_[kOuts];
  int n_outs_ = 0;
};

}  // namespace moert
