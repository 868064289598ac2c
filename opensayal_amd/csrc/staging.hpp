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

// up to here the layout kernels read and write a slot themselves; between
// kStagingShared and this only for a call that has the link to itself, since
// kernels of several threads share it worse than copies do (4 threads, fields
// of 1 MB in and out: 1550 us direct, 1290 through copies; one thread: 56 us in
// and 58 out, 62 and 59).  Below kStagingShared the runtime's copies are so much
// slower (0.52 MB in: 36 us, 236) that several threads lose nothing either.
constexpr size_t kStagingDirect = 1u << 20;
constexpr size_t kStagingShared = 1u << 19;
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
  // whether the layout kernels are to use the slot themselves
  bool direct(size_t bytes) const {
    return st_ && bytes <= (alone_ ? kStagingDirect : kStagingShared);
  }
  char* slot(size_t i = 0) const { return st_->host + i % kStagingSlots * kStagingSlot; }
  // dst <- src (device), after what `s` holds; dst is complete on return.
  // On an error nothing is in flight.
  hipError_t copy_out(void* dst, const void* src, size_t bytes, hipStream_t s);

 private:
  Staging* st_ = nullptr;
  bool alone_ = false;  // no other call had a buffer of the device when this took it
};

}  // namespace osy
