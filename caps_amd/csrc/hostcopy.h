// Copies between ordinary (pageable) host memory and the device, through a
// ring of pinned buffers.
//
// The runtime's own copy of pageable memory runs at 33 GB/s up and 18 GB/s
// down here (32 MiB), the DMA engines at 56 GB/s from pinned memory, one CPU
// thread's memcpy at 28-33 GB/s and four at 107 GB/s.  So a copy is cut into
// chunks: the calling thread, with a few helpers where they are worth it, moves
// pieces between the caller's memory and the ring while two streams move whole
// chunks between the ring and the device.
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>

namespace caps {

struct HostRange {
  void *dev;
  void *host;
  size_t bytes;
};

// Not thread safe; all streams and events belong to the device current at the
// first call.
class HostCopy {
 public:
  // host -> dev of every range; later work on s sees the data, the host memory
  // may be reused on return (as with hipMemcpyAsync of pageable memory).
  // Nothing else may be running on s.
  hipError_t up(const HostRange *r, int count, hipStream_t s);
  // dev -> host after the work on s; the data is there on return
  hipError_t down(const HostRange &r, hipStream_t s);
  void release();

 private:
  bool prepare();
  hipError_t send(const HostRange *r, int count, hipStream_t s);
  hipError_t receive(const HostRange &r, hipStream_t s);
  hipError_t settled(hipError_t e, hipStream_t s);
  static constexpr int SLOTS = 8;  // even: within a call a slot serves one stream
  char *ring_ = nullptr;
  hipStream_t side_ = nullptr;
  hipEvent_t landed_[SLOTS] = {};
  hipEvent_t order_ = nullptr;
};

}  // namespace caps
