// fake_hip.hpp - what the host paths see of fake_hip.cpp: a HIP runtime in
// host memory, and the solver's kernels as records of what was launched.
//
// A stream is a queue of pieces of work that run when something waits for it
// (or a test asks for a few of them).  A projection with the resident kernel
// is two pieces, its start and its end; in between its exchange buffer is in
// use, and whatever writes or frees that buffer then is a violation.  At its
// start the buffer must be live memory and hold empty words or what a launch
// of the same shape left.
#pragma once

#include <hip/hip_runtime.h>

#include <functional>
#include <string>
#include <vector>

#include "../../opensayal_amd/csrc/kernels.hpp"

namespace fake {

// A projection that was enqueued (or launched from a graph).
struct Launch {
  osy::ProjTuning tuning;
  int sweeps;
  bool resident;  // as one resident launch
  const void* exchange;
};

struct State {
  std::vector<std::string> violations;
  std::vector<Launch> launches;  // in the order they started
  size_t fail_malloc_from = ~size_t(0);  // hipMalloc of at least this many bytes fails
  long event_records_left = -1;  // hipEventRecord fails after as many (-1: never)
  int batch_launches = 0;
  int host_mallocs = 0, host_frees = 0;
  size_t device_bytes = 0;  // held by hipMalloc now
  // whether a resident launch of this shape times out
  std::function<bool(const osy::ProjTuning&)> times_out;
  // called in hipHostFree
  std::function<void()> on_host_free;
};

State& state();
// Runs the next `pieces` pieces of work of a stream.
void run(hipStream_t s, int pieces);
size_t pending(hipStream_t s);

}  // namespace fake
