// staging.hpp - pinned host memory for copies between pageable host memory
// and the device.
//
// A copy between the device and pageable memory goes through the runtime,
// which took 84 us for the 0.15 MB field of a 256 x 144 grid, 480 us for the
// 8.3 MB one of 1920 x 1080 and 1.9 ms at 3840 x 2160.  Here a kernel writes a
// field of up to kStagingDirect bytes into a pinned slot, or reads it from
// one (20 us), and larger results come through the slots in turn, a few
// threads copying from them, since what bounds a single one is reading memory
// that the device has just written, at 25 GB/s (1920 x 1080: 230 us, one
// thread 320; 3840 x 2160: 0.8 ms, one thread 1.2).  Larger fields go to
// the device through the runtime, which is as fast.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>

namespace osy {

// up to here the layout kernels read and write a slot themselves
constexpr size_t kStagingDirect = 1u << 20;
constexpr size_t kStagingSlot = 1u << 20;
constexpr int kStagingSlots = 4;

struct Staging {
  int device;
  char* host;  // kStagingSlots slots
  hipEvent_t done[kStagingSlots];
};

// Buffers are taken for the length of a call, so calls on several threads and
// streams never share one.  A device has at most kStagingKept of them, which
// are kept between calls; a call that finds them all taken goes without.  None
// is left once the last handle is gone.
constexpr int kStagingKept = 4;
void staging_retain();   // a handle is made
void staging_release();  // and destroyed

// A buffer for the call, when `host` is ordinary pageable memory (anything
// the runtime knows, it copies best by itself) and one can be had.
class StagingLease {
 public:
  StagingLease(int device, const void* host);
  ~StagingLease();
  StagingLease(const StagingLease&) = delete;
  StagingLease& operator=(const StagingLease&) = delete;
  explicit operator bool() const { return st_ != nullptr; }
  char* slot(size_t i = 0) const { return st_->host + i % kStagingSlots * kStagingSlot; }
  // dst <- src (device), after what `s` holds; dst is complete on return.
  // On an error nothing is in flight.
  hipError_t copy_out(void* dst, const void* src, size_t bytes, hipStream_t s);

 private:
  Staging* st_ = nullptr;
};

}  // namespace osy
