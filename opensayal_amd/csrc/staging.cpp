// staging.cpp - the pinned buffers of staging.hpp.
#include "staging.hpp"

#include <algorithm>
#include <cstring>
#include <exception>
#include <mutex>
#include <new>
#include <thread>

#include "kernels.hpp"

namespace osy {
namespace {

// The buffers of a device: `made` exist or are being made, `idle` of them lie
// here.
struct Pool {
  Staging* idle[kStagingKept];
  int idle_count, made;
};

constexpr int kMaxDevices = 64;
std::mutex g_mu;  // never held while one is made or freed
Pool g_pools[kMaxDevices];
long g_handles = 0;

void destroy(Staging* st) {
  for (hipEvent_t e : st->done)
    if (e) (void)hipEventDestroy(e);
  if (st->host) (void)hipHostFree(st->host);
  delete st;
}

Staging* create(int device) {
  int current = 0;
  if (hipGetDevice(&current) != hipSuccess) return nullptr;
  Staging* st = new (std::nothrow) Staging();
  if (!st) return nullptr;
  st->device = device;
  hipError_t e = current == device ? hipSuccess : hipSetDevice(device);
  if (e == hipSuccess)
    e = hipHostMalloc((void**)&st->host, kStagingSlots * kStagingSlot, hipHostMallocPortable);
  for (int i = 0; i < kStagingSlots && e == hipSuccess; i++)
    e = hipEventCreateWithFlags(&st->done[i], hipEventDisableTiming);
  if (current != device) (void)hipSetDevice(current);
  if (e != hipSuccess) {
    (void)hipGetLastError();  // the call goes on without
    destroy(st);
    return nullptr;
  }
  return st;
}

bool pageable(const void* host) {
  hipPointerAttribute_t a{};
  if (hipPointerGetAttributes(&a, host) != hipSuccess) {
    (void)hipGetLastError();
    return true;
  }
  return a.type == hipMemoryTypeUnregistered;
}

size_t chunk(size_t bytes, size_t i) {
  return std::min(kStagingSlot, bytes - i * kStagingSlot);
}

}  // namespace

void staging_retain() {
  std::lock_guard<std::mutex> lock(g_mu);
  g_handles++;
}

void staging_release() {
  for (Pool& pool : g_pools) {
    Staging* out[kStagingKept];
    int n = 0;
    {
      std::lock_guard<std::mutex> lock(g_mu);
      if (&pool == g_pools) g_handles--;
      if (g_handles > 0) return;
      n = pool.idle_count;
      std::copy(pool.idle, pool.idle + n, out);
      pool.idle_count = 0;
      pool.made -= n;
    }
    for (int i = 0; i < n; i++) destroy(out[i]);
  }
}

StagingLease::StagingLease(int device, const void* host) {
  if (!host || device < 0 || device >= kMaxDevices || !pageable(host)) return;
  Pool& pool = g_pools[device];
  {
    std::lock_guard<std::mutex> lock(g_mu);
    alone_ = pool.made == pool.idle_count;
    if (pool.idle_count > 0) {
      st_ = pool.idle[--pool.idle_count];
      return;
    }
    if (pool.made == kStagingKept) return;  // all are out: the runtime's copy
    pool.made++;
  }
  st_ = create(device);
  if (st_) return;
  std::lock_guard<std::mutex> lock(g_mu);
  pool.made--;
}

StagingLease::~StagingLease() {
  if (!st_) return;
  Pool& pool = g_pools[st_->device];
  {
    std::lock_guard<std::mutex> lock(g_mu);
    if (g_handles > 0) {
      pool.idle[pool.idle_count++] = st_;
      return;
    }
    pool.made--;
  }
  destroy(st_);
}

hipError_t StagingLease::copy_out(void* dst, const void* src, size_t bytes, hipStream_t s) {
  const size_t n = (bytes + kStagingSlot - 1) / kStagingSlot;
  auto issue = [&](size_t i) {
    enqueue_copy(slot(i), (const char*)src + i * kStagingSlot, (chunk(bytes, i) + 15) / 16 * 16,
                 s);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? hipEventRecord(st_->done[i % kStagingSlots], s) : e;
  };
  // chunks t, t + threads, ... (a slot belongs to one thread)
  auto take = [&](size_t t, size_t threads) {
    hipError_t e = hipSuccess;
    for (size_t i = t; i < n && e == hipSuccess; i += threads) {
      e = hipEventSynchronize(st_->done[i % kStagingSlots]);
      if (e != hipSuccess) break;
      std::memcpy((char*)dst + i * kStagingSlot, slot(i), chunk(bytes, i));
      if (i + kStagingSlots < n) e = issue(i + kStagingSlots);
    }
    return e;
  };
  hipError_t e = hipSuccess;
  for (size_t i = 0; i < std::min<size_t>(n, kStagingSlots) && e == hipSuccess; i++) e = issue(i);
  if (e == hipSuccess) {
    const size_t threads = n < 4 ? 1 : kStagingSlots;
    hipError_t helped[kStagingSlots] = {};
    std::thread helper[kStagingSlots];
    for (size_t t = 1; t < threads; t++) {
      try {
        helper[t] = std::thread([&, t] {
          helped[t] = hipSetDevice(st_->device);
          if (helped[t] == hipSuccess) helped[t] = take(t, threads);
        });
      } catch (const std::exception&) {  // no thread to be had: this one takes its part
        helped[t] = take(t, threads);
      }
    }
    e = take(0, threads);
    for (size_t t = 1; t < threads; t++) {
      if (helper[t].joinable()) helper[t].join();
      if (e == hipSuccess) e = helped[t];
    }
  }
  if (e != hipSuccess) (void)hipStreamSynchronize(s);
  return e;
}

}  // namespace osy
