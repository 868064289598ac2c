#include "fake_hip.hpp"

#include <cstdlib>
#include <cstring>
#include <deque>
#include <map>
#include <memory>
#include <mutex>

#include "../../opensayal_amd/csrc/batch.hpp"

using namespace osy;

namespace {

using Work = std::function<void()>;

struct Stream {
  std::deque<Work> queue;
  std::vector<Work>* capture = nullptr;
};
struct Event {
  double at = 0;
};
struct Graph {
  std::vector<Work> work;
};
struct Alloc {
  size_t bytes;
  int in_use;
};

std::recursive_mutex g_mu;
std::map<char*, Alloc> g_live;
std::vector<Stream*> g_streams;
double g_clock = 0;  // ms
thread_local hipError_t t_last = hipSuccess;

#define LOCK std::lock_guard<std::recursive_mutex> lock(g_mu)

hipError_t done(hipError_t e) {
  if (e != hipSuccess) t_last = e;
  return e;
}

void violation(const std::string& what) { fake::state().violations.push_back(what); }

std::map<char*, Alloc>::iterator holder(const void* p) {
  auto it = g_live.upper_bound((char*)p);
  if (it == g_live.begin()) return g_live.end();
  --it;
  return (char*)p < it->first + it->second.bytes ? it : g_live.end();
}

// a write by anything but the launch that uses the memory
void writes(const void* p, const char* who) {
  auto it = holder(p);
  if (it != g_live.end() && it->second.in_use)
    violation(std::string(who) + " while a resident launch uses the exchange buffer");
}

Stream* of(hipStream_t s) { return (Stream*)s; }

void drain(Stream* s) {
  while (s && !s->queue.empty()) {
    Work w = std::move(s->queue.front());
    s->queue.pop_front();
    w();
  }
}
void drain_all() {
  for (size_t i = 0; i < g_streams.size(); i++) drain(g_streams[i]);
}

void push(hipStream_t s, Work w) {
  LOCK;
  if (!s) {
    w();
  } else if (of(s)->capture) {
    of(s)->capture->push_back(std::move(w));
  } else {
    of(s)->queue.push_back(std::move(w));
  }
}

// ---- the projection ----------------------------------------------------------

unsigned long long tag_of(const ProjTuning& t) {
  return 1000ULL * t.k + t.reg_rows();
}
constexpr unsigned long long kClean = ~0ULL, kHalfRead = 7;

void project(const StepParams& sp, const FieldPtrs& f, const ProjTuning& t, size_t elem,
             hipStream_t s) {
  if (sp.n <= 0) return;
  ProjTuning run;
  const bool resident = t.kernel == PROJ_RESIDENT && f.exchange &&
                        t.resident_plan(sp.W, sp.H, sp.cus, &run);
  auto& st = fake::state();
  if (!resident) {
    push(s, [=, &st] {
      st.launches.push_back({t, sp.n, false, nullptr});
      g_clock += 10.0 + 0.01 * t.k;
    });
    return;
  }
  const size_t bytes = 3 * 8 * run.exchange_words(sp.W, sp.H, elem);
  push(s, [=, &st] {
    st.launches.push_back({t, sp.n, true, f.exchange});
    auto it = holder(f.exchange);
    if (it == g_live.end() || holder((char*)f.exchange + bytes - 1) != it ||
        holder(f.rstate) != it) {
      violation("a resident launch on memory that is not held");
      return;
    }
    unsigned long long tag;
    std::memcpy(&tag, f.exchange, 8);
    if (tag != kClean && tag != tag_of(run) && *f.error == 0)
      violation("a resident launch found words that another shape or a timed-out wait left");
    it->second.in_use++;
  });
  push(s, [=, &st] {
    auto it = holder(f.exchange);
    if (it == g_live.end()) return;
    it->second.in_use--;
    unsigned long long tag = tag_of(run);
    if (*f.error != 0) {
      tag = kHalfRead;  // it left without waiting
      g_clock += 0.001;
    } else if (st.times_out && st.times_out(t)) {
      tag = kHalfRead;
      *f.error = 1;
      g_clock += 2000.0;
    } else {
      g_clock += 5.0;
    }
    std::memcpy(f.exchange, &tag, 8);
  });
}

}  // namespace

namespace fake {
State& state() {
  static State s;
  return s;
}
void run(hipStream_t s, int pieces) {
  LOCK;
  for (int i = 0; i < pieces && !of(s)->queue.empty(); i++) {
    Work w = std::move(of(s)->queue.front());
    of(s)->queue.pop_front();
    w();
  }
}
size_t pending(hipStream_t s) {
  LOCK;
  return of(s)->queue.size();
}
}  // namespace fake

// ---- kernels ---------------------------------------------------------------------

namespace osy {

hipError_t init_projection_kernels() { return hipSuccess; }
void launch_build_flags(const MaskParams&, uint8_t*, uint8_t*, hipStream_t) {}

void enqueue_step(int storage, const StepParams& sp, const FieldPtrs& f, int* uv, int* sm,
                  const ProjTuning& t, hipStream_t s) {
  project(sp, f, t, storage == OSY_STORAGE_F32 ? 4 : 2, s);
  *uv = 1 - *uv;
  if (sp.smoke_on) *sm = 1 - *sm;
}
void enqueue_projection_only(int storage, const StepParams& sp, const FieldPtrs& f, int* uv,
                             const ProjTuning& t, hipStream_t s) {
  project(sp, f, t, storage == OSY_STORAGE_F32 ? 4 : 2, s);
  *uv = 1 - *uv;
}
void enqueue_divergence(int, const StepParams&, const FieldPtrs&, int, hipStream_t) {}
void enqueue_export(int, int, const StepParams&, const FieldPtrs&, int, int, void*, hipStream_t) {}
void enqueue_import(int, int, const StepParams&, const FieldPtrs&, int, int, const void*,
                    hipStream_t) {}
void enqueue_render(int, const StepParams&, const FieldPtrs&, int, int, int, uint32_t*,
                    hipStream_t) {}
void enqueue_traces(int, const StepParams&, const FieldPtrs&, int, int, int, float, int32_t*,
                    int32_t*, hipStream_t) {}
void enqueue_copy(void* dst, const void* src, size_t bytes, hipStream_t s) {
  push(s, [=] { std::memcpy(dst, src, bytes); });
}
void enqueue_clean_exchange(void* mem, size_t bytes, hipStream_t s) {
  push(s, [=] {
    writes(mem, "cleaning");
    std::memset(mem, 0, 256);
    std::memset((char*)mem + 256, 0xFF, bytes - 256);
  });
}
void enqueue_pressure_range(const StepParams&, const FieldPtrs&, hipStream_t) {}
hipError_t batch_grid_size(int, bool, int, int, int* grid) {
  *grid = 256;
  return hipSuccess;
}
void enqueue_batch_step(int, bool, int, int, const BatchArgs&, hipStream_t s) {
  push(s, [] { fake::state().batch_launches++; });
}

}  // namespace osy

// ---- the runtime ---------------------------------------------------------------

extern "C" {

hipError_t hipGetLastError(void) {
  const hipError_t e = t_last;
  t_last = hipSuccess;
  return e;
}
const char* hipGetErrorString(hipError_t e) {
  return e == hipErrorOutOfMemory ? "out of memory" : "an error";
}
hipError_t hipGetDevice(int* d) {
  *d = 0;
  return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDeviceCount(int* n) {
  *n = 1;
  return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t a, int) {
  *v = a == hipDeviceAttributeMultiprocessorCount ? 256 : 100000;
  return hipSuccess;
}
hipError_t hipMalloc(void** p, size_t bytes) {
  LOCK;
  if (bytes >= fake::state().fail_malloc_from) {
    *p = (void*)0x40;  // what a failed call leaves there is not for use
    return done(hipErrorOutOfMemory);
  }
  *p = std::calloc(1, bytes);
  g_live[(char*)*p] = {bytes, 0};
  fake::state().device_bytes += bytes;
  return hipSuccess;
}
hipError_t hipFree(void* p) {
  LOCK;
  if (!p) return hipSuccess;
  drain_all();  // hipFree waits for the device
  auto it = g_live.find((char*)p);
  if (it == g_live.end()) {
    violation("hipFree of memory that is not held");
    return done(hipErrorInvalidValue);
  }
  fake::state().device_bytes -= it->second.bytes;
  g_live.erase(it);
  std::free(p);
  return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t bytes, unsigned) {
  LOCK;
  fake::state().host_mallocs++;
  *p = std::malloc(bytes);
  return hipSuccess;
}
hipError_t hipHostFree(void* p) {
  if (fake::state().on_host_free) fake::state().on_host_free();
  LOCK;
  fake::state().host_frees++;
  std::free(p);
  return hipSuccess;
}
hipError_t hipPointerGetAttributes(hipPointerAttribute_t*, const void*) {
  return done(hipErrorInvalidValue);  // ordinary memory
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) {
  LOCK;
  writes(d, "a copy");
  std::memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind kind, hipStream_t st) {
  LOCK;
  if (kind == hipMemcpyHostToDevice && st && !of(st)->capture) drain(of(st));
  auto copy = [=] {
    writes(d, "a copy");
    std::memcpy(d, s, n);
  };
  if (kind == hipMemcpyHostToDevice && st && !of(st)->capture)
    copy();
  else
    push(st, copy);
  return hipSuccess;
}
hipError_t hipMemset(void* d, int v, size_t n) {
  LOCK;
  std::memset(d, v, n);
  return hipSuccess;
}
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t s) {
  LOCK;
  if (s && of(s)->capture) violation("hipMemsetAsync in a captured graph");
  push(s, [=] {
    writes(d, "a fill");
    std::memset(d, v, n);
  });
  return hipSuccess;
}
hipError_t hipDeviceSynchronize(void) {
  LOCK;
  drain_all();
  return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
  LOCK;
  Stream* n = new Stream;
  g_streams.push_back(n);
  *s = (hipStream_t)n;
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) {
  LOCK;
  drain(of(s));
  for (size_t i = 0; i < g_streams.size(); i++)
    if (g_streams[i] == of(s)) g_streams.erase(g_streams.begin() + i);
  delete of(s);
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t s) {
  LOCK;
  drain(of(s));
  return hipSuccess;
}
hipError_t hipStreamIsCapturing(hipStream_t s, hipStreamCaptureStatus* c) {
  LOCK;
  *c = s && of(s)->capture ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
  return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t s, hipStreamCaptureMode) {
  LOCK;
  of(s)->capture = new std::vector<Work>;
  return hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t s, hipGraph_t* g) {
  LOCK;
  Graph* n = new Graph{std::move(*of(s)->capture)};
  delete of(s)->capture;
  of(s)->capture = nullptr;
  *g = (hipGraph_t)n;
  return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t* x, hipGraph_t g, hipGraphNode_t*, char*, size_t) {
  LOCK;
  *x = (hipGraphExec_t) new Graph(*(Graph*)g);
  return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t x, hipStream_t s) {
  LOCK;
  for (const Work& w : ((Graph*)x)->work) push(s, w);
  return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t g) {
  delete (Graph*)g;
  return hipSuccess;
}
hipError_t hipGraphExecDestroy(hipGraphExec_t x) {
  delete (Graph*)x;
  return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t* e) {
  *e = (hipEvent_t) new Event;
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e) {
  delete (Event*)e;
  return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  long& left = fake::state().event_records_left;
  if (left == 0) return done(hipErrorUnknown);
  if (left > 0) left--;
  push(s, [e] { ((Event*)e)->at = g_clock; });
  return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t) {
  LOCK;
  drain_all();
  return hipSuccess;
}
hipError_t hipEventElapsedTime(float* ms, hipEvent_t a, hipEvent_t z) {
  *ms = (float)(((Event*)z)->at - ((Event*)a)->at);
  return hipSuccess;
}

}  // extern "C"
