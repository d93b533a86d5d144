// transfer.h -- copies between pageable host arrays and the device through
// pinned chunks that several threads fill or empty (internal to the library).
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <memory>

namespace colphys {

// One engine serves a handle (an ensemble's members share their parent's)
// and goes with it; one transfer runs at a time.  Four pinned chunks of
// 4 MiB (16 after a transfer of 64 MiB and more) and up to seven threads are
// made at the first large transfer.  The threads are asleep but for some tens
// of microseconds at the start of a transfer and after a chunk: the calling
// thread alone waits for the work that the stream holds.
//
// hipMemcpy on pageable memory copies through the runtime's own pinned
// buffer with the calling thread alone.  That thread's memcpy bounds it, and
// on the way to the host its page faults in a fresh destination.
class Transfer {
 public:
  Transfer();
  ~Transfer();
  Transfer(const Transfer&) = delete;
  Transfer& operator=(const Transfer&) = delete;
  // Device to host and host to device, ordered after the stream's work.
  // to_host returns when dst is written, to_device when src has been read
  // (the last chunks may still be on their way in the stream's order).
  hipError_t to_host(void* dst, const void* dev, size_t bytes, hipStream_t stream);
  hipError_t to_device(void* dev, const void* src, size_t bytes, hipStream_t stream);
  // Host to host.
  void copy(void* dst, const void* src, size_t bytes);

 private:
  struct Impl;
  std::unique_ptr<Impl> im_;
};

}  // namespace colphys
