// host_paths.cpp - the host side of the solver (fluid_host.cpp, batch_host.cpp,
// staging.cpp) on a runtime in host memory (fake_hip.cpp): what happens to
// device memory and streams where a GPU could only fault.  One scenario per
// run, named by the first argument; prints "ok", or what went wrong.
#include <chrono>
#include <cstdio>
#include <cstring>
#include <future>
#include <map>
#include <memory>
#include <string>
#include <vector>

#include "../../include/opensayal.h"
#include "../../opensayal_amd/csrc/staging.hpp"
#include "fake_hip.hpp"

namespace {

int g_failed = 0;

void expect(bool ok, const char* what) {
  if (ok) return;
  std::printf("failed: %s\n", what);
  g_failed = 1;
}
#define EXPECT(x) expect((x), #x)

osy_config config(int W, int H, int n, bool pressure = false) {
  osy_config c;
  osy_config_defaults(&c);
  char text[128];
  std::snprintf(text, sizeof text,
                "{\"sim\": {\"width\": %d, \"height\": %d}, \"fluid\": {\"viscosity\": 0}}", W, H);
  osy_config_parse_string(text, &c);
  c.projection_n = n;
  c.enable_pressure = pressure ? 1 : 0;
  return c;
}

osy_fluid* create(const osy_config& c) {
  osy_fluid* fl = nullptr;
  EXPECT(osy_fluid_create(&c, &fl) == OSY_OK);
  return fl;
}

// A register (2) or resident (3) shape of `rows` x 8 region rows.
osy_tuning shape(int kernel, int rows, int k) {
  osy_tuning t;
  t.projection_kernel = kernel;
  t.tile_width = 128 - 4 * k;
  t.tile_height = 8 * rows - 4 * k;
  t.sweeps_per_launch = k;
  return t;
}

// A larger exchange buffer cannot be had: the shape is refused, and the
// handle goes on with what it has.
void exchange_out_of_memory() {
  osy_fluid* fl = create(config(250, 230, 20));
  osy_tuning small = shape(3, 12, 5), large = shape(3, 4, 3);
  EXPECT(osy_fluid_set_tuning(fl, &small) == OSY_OK);
  EXPECT(osy_fluid_step(fl, 5, 0.05f) == OSY_OK);
  fake::state().fail_malloc_from = 1;
  EXPECT(osy_fluid_set_tuning(fl, &large) == OSY_E_NOMEM);
  // no error is left behind for the calls that follow
  EXPECT(osy_fluid_project(fl, 20, nullptr) == OSY_OK);
  EXPECT(osy_fluid_step(fl, 5, 0.05f) == OSY_OK);
  osy_tuning now;
  EXPECT(osy_fluid_get_tuning(fl, &now) == OSY_OK);
  EXPECT(std::memcmp(&now, &small, sizeof now) == 0);
  fake::state().fail_malloc_from = ~size_t(0);
  EXPECT(osy_fluid_set_tuning(fl, &large) == OSY_OK);
  EXPECT(osy_fluid_step(fl, 5, 0.05f) == OSY_OK);
  EXPECT(fake::state().launches.back().resident);
  osy_fluid_destroy(fl);
}

// An autotune that fails on the way leaves the handle, its exchange buffer and
// the graphs that name it as they were.
void autotune_fails() {
  osy_fluid* fl = create(config(250, 230, 20));
  osy_tuning mine = shape(3, 12, 5);
  EXPECT(osy_fluid_set_tuning(fl, &mine) == OSY_OK);
  for (int parity = 0; parity < 2; parity++) EXPECT(osy_fluid_step(fl, 5, 0.05f) == OSY_OK);
  for (long records = 1; records < 700; records += 3) {
    fake::state().event_records_left = records;
    const int st = osy_fluid_autotune(fl, nullptr, nullptr);
    if (st == OSY_OK) break;  // there were enough
    fake::state().event_records_left = -1;
    EXPECT(osy_fluid_step(fl, 5, 0.05f) == OSY_OK);
    osy_tuning now;
    EXPECT(osy_fluid_get_tuning(fl, &now) == OSY_OK);
    EXPECT(std::memcmp(&now, &mine, sizeof now) == 0);
  }
  osy_fluid_destroy(fl);
  EXPECT(fake::state().device_bytes == 0);
}

// No memory for any exchange buffer: the autotuner picks among the others.
void autotune_without_exchange() {
  osy_fluid* fl = create(config(250, 230, 20));
  fake::state().fail_malloc_from = 1 << 20;  // the snapshot fits
  osy_tuning best;
  EXPECT(osy_fluid_autotune(fl, &best, nullptr) == OSY_OK);
  EXPECT(best.projection_kernel != 3);
  EXPECT(osy_fluid_step(fl, 5, 0.05f) == OSY_OK);
  osy_fluid_destroy(fl);
}

// A resident trial whose wait times out leaves early from then on; its time is
// no time of that shape, nor are the ones after it.
void autotune_times_out() {
  osy_tuning best;
  osy_fluid* one = create(config(250, 230, 20));
  fake::state().times_out = [](const osy::ProjTuning& t) { return t.k == 5; };
  EXPECT(osy_fluid_autotune(one, &best, nullptr) == OSY_OK);
  EXPECT(best.projection_kernel == 3 && best.sweeps_per_launch != 5);
  EXPECT(osy_fluid_step(one, 5, 0.05f) == OSY_OK);
  osy_fluid_destroy(one);
  osy_fluid* all = create(config(250, 231, 20));
  fake::state().times_out = [](const osy::ProjTuning&) { return true; };
  EXPECT(osy_fluid_autotune(all, &best, nullptr) == OSY_OK);
  EXPECT(best.projection_kernel != 3);
  osy_fluid* next = create(config(250, 231, 20));
  EXPECT(osy_fluid_autotune_cached(next) == 1);
  EXPECT(osy_fluid_get_tuning(next, &best) == OSY_OK);
  EXPECT(best.projection_kernel != 3);
  EXPECT(osy_fluid_step(all, 5, 0.05f) == OSY_OK);
  EXPECT(osy_fluid_synchronize(all) == OSY_OK);
  osy_fluid_destroy(next);
  osy_fluid_destroy(all);
}

// A wait that times out in a batch autotuner's trial, in a member that steps
// on its own graphs: its state is put back, and its rings are clean again.
void batch_autotune_times_out() {
  osy_fluid* own = create(config(250, 230, 20));
  osy_fluid* shared = create(config(64, 36, 20));
  osy_batch* b = nullptr;
  EXPECT(osy_batch_create(0, &b) == OSY_OK);
  EXPECT(osy_batch_set_per_grid_cells(b, 250 * 230) == OSY_OK);
  EXPECT(osy_batch_add(b, own) == OSY_OK);
  EXPECT(osy_batch_add(b, shared) == OSY_OK);
  fake::state().times_out = [](const osy::ProjTuning&) {
    return fake::state().batch_launches == 100;
  };
  EXPECT(osy_batch_autotune(b, nullptr, nullptr) == OSY_OK);
  EXPECT(fake::state().batch_launches > 100);
  fake::state().times_out = nullptr;
  osy_tuning t;
  EXPECT(osy_fluid_get_tuning(own, &t) == OSY_OK && t.projection_kernel == 3);
  fake::state().violations.clear();  // those of the trials, whose results are dropped
  EXPECT(osy_batch_step(b, 4) == OSY_OK);
  float p[250 * 230];
  EXPECT(osy_fluid_get_field(own, OSY_FIELD_VEL_X, p, sizeof p) == OSY_OK);
  osy_batch_destroy(b);
  osy_fluid_destroy(own);
  osy_fluid_destroy(shared);
}

// The exchange buffer is cleaned in the order of the stream that uses it: not
// while a launch that the caller put on a stream of their own is running.
void cleaned_in_stream_order() {
  osy_fluid* fl = create(config(250, 230, 20));
  osy_tuning first = shape(3, 12, 5), second = shape(3, 12, 4);
  void* s = nullptr;
  EXPECT(osy_stream_create(&s) == OSY_OK);
  EXPECT(osy_fluid_set_tuning(fl, &second) == OSY_OK);
  EXPECT(osy_fluid_set_tuning(fl, &first) == OSY_OK);
  EXPECT(osy_fluid_step_async(fl, 2, 0.05f, s) == OSY_OK);
  while (fake::state().launches.empty()) fake::run((hipStream_t)s, 1);
  // the first step's launch is running
  EXPECT(fake::state().launches.size() == 1);
  EXPECT(osy_fluid_set_tuning(fl, &second) == OSY_OK);
  EXPECT(osy_fluid_step_async(fl, 3, 0.05f, s) == OSY_OK);
  EXPECT(osy_stream_synchronize(s) == OSY_OK);
  EXPECT(fake::state().launches.size() == 5);

  fake::state().times_out = [](const osy::ProjTuning&) {
    return fake::state().launches.size() == 6;
  };
  EXPECT(osy_fluid_step_async(fl, 2, 0.05f, s) == OSY_OK);
  while (fake::state().launches.size() < 7) fake::run((hipStream_t)s, 1);
  // the sixth has timed out, the seventh is running
  EXPECT(osy_fluid_synchronize(fl) == OSY_E_STATE);
  EXPECT(osy_fluid_step_async(fl, 2, 0.05f, s) == OSY_OK);
  EXPECT(osy_stream_synchronize(s) == OSY_OK);
  EXPECT(fake::state().launches.size() == 9);
  EXPECT(osy_fluid_synchronize(fl) == OSY_OK);
  osy_fluid_destroy(fl);
  EXPECT(osy_stream_destroy(s) == OSY_OK);
}

// A projection that the caller captured goes on working with its own exchange
// buffer, whatever shapes the handle takes after that.
void captured_projection() {
  osy_fluid* fl = create(config(250, 230, 20));
  const osy_tuning first = shape(3, 12, 5), larger = shape(3, 4, 3), smaller = shape(3, 12, 4),
                   launches = shape(2, 8, 5);
  void* s = nullptr;
  EXPECT(osy_stream_create(&s) == OSY_OK);
  EXPECT(osy_fluid_set_tuning(fl, &first) == OSY_OK);
  hipGraph_t graph = nullptr;
  hipGraphExec_t exec = nullptr;
  EXPECT(hipStreamBeginCapture((hipStream_t)s, hipStreamCaptureModeThreadLocal) == hipSuccess);
  for (int i = 0; i < 2; i++) EXPECT(osy_fluid_project(fl, 20, s) == OSY_OK);
  EXPECT(hipStreamEndCapture((hipStream_t)s, &graph) == hipSuccess);
  EXPECT(hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0) == hipSuccess);
  size_t held = 0;
  for (int round = 0; round < 3; round++) {
    for (const osy_tuning* t : {&larger, &smaller, &launches, &first}) {
      EXPECT(osy_fluid_set_tuning(fl, t) == OSY_OK);
      EXPECT(osy_fluid_step_async(fl, 2, 0.05f, s) == OSY_OK);
      EXPECT(hipGraphLaunch(exec, (hipStream_t)s) == hipSuccess);
      EXPECT(osy_fluid_step_async(fl, 2, 0.05f, s) == OSY_OK);
      EXPECT(osy_stream_synchronize(s) == OSY_OK);
      EXPECT(osy_fluid_synchronize(fl) == OSY_OK);
    }
    if (round == 1) held = fake::state().device_bytes;
    if (round == 2) EXPECT(fake::state().device_bytes == held);
  }
  // one of its replays times out while the handle has another shape
  EXPECT(osy_fluid_set_tuning(fl, &smaller) == OSY_OK);
  EXPECT(osy_fluid_step_async(fl, 2, 0.05f, s) == OSY_OK);
  EXPECT(osy_stream_synchronize(s) == OSY_OK);
  EXPECT(osy_fluid_synchronize(fl) == OSY_OK);
  fake::state().times_out = [](const osy::ProjTuning& t) { return t.k == 5; };
  EXPECT(hipGraphLaunch(exec, (hipStream_t)s) == hipSuccess);
  EXPECT(osy_stream_synchronize(s) == OSY_OK);
  fake::state().times_out = nullptr;
  EXPECT(osy_fluid_synchronize(fl) == OSY_E_STATE);
  EXPECT(hipGraphLaunch(exec, (hipStream_t)s) == hipSuccess);
  EXPECT(osy_stream_synchronize(s) == OSY_OK);
  EXPECT(osy_fluid_synchronize(fl) == OSY_OK);
  hipGraphExecDestroy(exec);
  hipGraphDestroy(graph);
  osy_fluid_destroy(fl);
  EXPECT(osy_stream_destroy(s) == OSY_OK);
  EXPECT(fake::state().device_bytes == 0);
}

uint64_t device_bytes(osy_fluid* fl) {
  osy_fluid_info info;
  EXPECT(osy_fluid_get_info(fl, &info) == OSY_OK);
  return info.device_bytes;
}

// The exchange buffer is part of the device memory a handle says it holds, and
// goes when another kernel is chosen.
void exchange_is_counted() {
  osy_fluid* fl = create(config(250, 230, 20));
  const uint64_t plain = device_bytes(fl);
  EXPECT(plain == fake::state().device_bytes);
  const osy_tuning resident = shape(3, 12, 5), launches = shape(2, 8, 5);
  EXPECT(osy_fluid_set_tuning(fl, &resident) == OSY_OK);
  EXPECT(device_bytes(fl) > plain);
  EXPECT(device_bytes(fl) == fake::state().device_bytes);
  EXPECT(osy_fluid_step(fl, 4, 0.05f) == OSY_OK);
  EXPECT(osy_fluid_set_tuning(fl, &launches) == OSY_OK);
  EXPECT(device_bytes(fl) == plain);
  EXPECT(fake::state().device_bytes == plain);
  EXPECT(osy_fluid_step(fl, 4, 0.05f) == OSY_OK);
  osy_fluid_destroy(fl);
}

// A batch's budget bounds its members' exchange buffers too: what does not
// fit is given back, and the autotuner does not pick what would not.
void exchange_in_a_budget() {
  const osy_config c = config(250, 230, 20);
  uint64_t plain = 0;
  EXPECT(osy_fluid_device_bytes(&c, &plain) == OSY_OK);
  const osy_tuning resident = shape(3, 12, 5);
  for (const uint64_t budget : {2 * plain + 100000, uint64_t(1) << 32}) {
    const bool fits = budget > 3 * plain;
    osy_fluid *one = create(c), *two = create(c);
    EXPECT(osy_fluid_set_tuning(one, &resident) == OSY_OK);
    for (int parity = 0; parity < 2; parity++) EXPECT(osy_fluid_step(one, 5, 0.05f) == OSY_OK);
    osy_batch* b = nullptr;
    osy_batch_info info;
    EXPECT(osy_batch_create(budget, &b) == OSY_OK);
    EXPECT(osy_batch_set_per_grid_cells(b, 1) == OSY_OK);
    EXPECT(osy_batch_add(b, one) == OSY_OK);
    EXPECT(osy_batch_add(b, two) == OSY_OK);
    EXPECT(osy_batch_step(b, 2) == OSY_OK);
    EXPECT(!fake::state().launches.back().resident);  // member two
    EXPECT((fake::state().launches.end() - 2)->resident == fits);
    EXPECT(osy_batch_get_info(b, &info) == OSY_OK);
    EXPECT(info.used_bytes == device_bytes(one) + device_bytes(two));
    EXPECT(info.used_bytes <= budget);
    EXPECT(osy_batch_autotune(b, nullptr, nullptr) == OSY_OK);
    EXPECT(osy_batch_get_info(b, &info) == OSY_OK);
    EXPECT(info.used_bytes == device_bytes(one) + device_bytes(two));
    EXPECT(info.used_bytes <= budget);
    EXPECT((info.used_bytes > 2 * plain) == fits);
    EXPECT(osy_batch_step(b, 2) == OSY_OK);
    osy_fluid* three = create(c);
    EXPECT(osy_batch_add(b, three) == (fits ? OSY_OK : OSY_E_BUDGET));
    osy_batch_destroy(b);
    for (osy_fluid* fl : {one, two, three}) osy_fluid_destroy(fl);
  }
  EXPECT(fake::state().device_bytes == 0);
}

// A resident shape that runs as a launch per stage says so.
void resident_says_what_runs() {
  osy_fluid* fl = create(config(2400, 1400, 20));
  // 500 tiles of 64 rows, which the call takes; 320 of 96, which do not fit
  const osy_tuning asked = shape(3, 8, 2), fits = shape(3, 12, 5);
  osy_fluid_info info;
  osy_tuning now;
  EXPECT(osy_fluid_set_tuning(fl, &asked) == OSY_OK);
  EXPECT(osy_fluid_project(fl, 20, nullptr) == OSY_OK);
  EXPECT(osy_fluid_synchronize(fl) == OSY_OK);
  EXPECT(!fake::state().launches.back().resident);
  EXPECT(osy_fluid_get_info(fl, &info) == OSY_OK);
  EXPECT(info.projection_kernel == 2 && info.sweeps_per_launch == 2);
  EXPECT(osy_fluid_get_tuning(fl, &now) == OSY_OK);
  EXPECT(std::memcmp(&now, &asked, sizeof now) == 0);
  EXPECT(osy_fluid_set_tuning(fl, &fits) == OSY_E_INVALID);  // 414 tiles
  osy_fluid_destroy(fl);
  fl = create(config(1920, 1080, 20));
  EXPECT(osy_fluid_set_tuning(fl, &fits) == OSY_OK);
  EXPECT(osy_fluid_project(fl, 20, nullptr) == OSY_OK);
  EXPECT(osy_fluid_synchronize(fl) == OSY_OK);
  EXPECT(fake::state().launches.back().resident);
  EXPECT(osy_fluid_get_info(fl, &info) == OSY_OK);
  EXPECT(info.projection_kernel == 3 && info.sweeps_per_launch == 5);
  osy_fluid_destroy(fl);
}

// One whose pressure sums divide (d_t = 0 or |d_t| >= 2) is resident like the
// others.
void dividing_is_resident() {
  for (const float d_t : {0.05f, 0.0f, 2.0f, -3.5f}) {
    osy_config c = config(250, 230, 20, true);
    c.d_t = d_t;
    osy_fluid* fl = create(c);
    const osy_tuning asked = shape(3, 8, 5);
    osy_fluid_info info;
    EXPECT(osy_fluid_set_tuning(fl, &asked) == OSY_OK);
    EXPECT(osy_fluid_project(fl, 20, nullptr) == OSY_OK);
    EXPECT(osy_fluid_synchronize(fl) == OSY_OK);
    EXPECT(fake::state().launches.back().resident);
    EXPECT(osy_fluid_get_info(fl, &info) == OSY_OK);
    EXPECT(info.projection_kernel == 3);
    osy_fluid_destroy(fl);
  }
}

// Pinned buffers are made a few times per device and kept, however many callers
// there are, and nobody waits while one is freed.
void staging_is_bounded() {
  using osy::StagingLease;
  char host[16];
  osy::staging_retain();
  for (int round = 0; round < 3; round++) {
    std::vector<std::unique_ptr<StagingLease>> at_once;
    for (int i = 0; i < 7; i++) at_once.emplace_back(new StagingLease(0, host));
    int have = 0;
    for (auto& lease : at_once) have += *lease ? 1 : 0;
    EXPECT(have == osy::kStagingKept);
  }
  EXPECT(fake::state().host_mallocs == osy::kStagingKept);
  for (int round = 0; round < 3; round++)
    for (int device = 1; device < 8; device++) EXPECT((bool)StagingLease(device, host));
  EXPECT(fake::state().host_mallocs == osy::kStagingKept + 7);
  EXPECT(fake::state().host_frees == 0);
  std::vector<std::future<void>> others;
  fake::state().on_host_free = [&] {
    if (!others.empty()) return;
    others.push_back(std::async(std::launch::async, [&host] { StagingLease lease(9, host); }));
    EXPECT(others.back().wait_for(std::chrono::seconds(2)) == std::future_status::ready);
  };
  osy::staging_release();
  others.clear();
  EXPECT(fake::state().host_frees == fake::state().host_mallocs);
}

// The layout kernels use a slot for larger fields only in a call that has the
// device's link to itself.
void staging_shares_the_link() {
  using osy::StagingLease;
  char host[16];
  osy::staging_retain();
  for (int round = 0; round < 3; round++) {
    StagingLease first(0, host);
    EXPECT(first.direct(osy::kStagingDirect) && !first.direct(osy::kStagingDirect + 1));
    StagingLease second(0, host), elsewhere(1, host);
    EXPECT(second.direct(osy::kStagingShared) && !second.direct(osy::kStagingShared + 1));
    EXPECT(elsewhere.direct(osy::kStagingDirect));
  }
  EXPECT(!StagingLease(0, nullptr).direct(4));  // no buffer
  osy::staging_release();
}

// Members whose pressure sums divide (d_t = 0 or |d_t| >= 2) step in the
// batch's launch like the others.
void batch_division() {
  osy_batch* b = nullptr;
  EXPECT(osy_batch_create(0, &b) == OSY_OK);
  std::vector<osy_fluid*> members;
  for (const float d_t : {0.05f, 0.0f, 2.0f, -3.5f}) {
    osy_config c = config(64, 36, 20, true);
    c.d_t = d_t;
    members.push_back(create(c));
    EXPECT(osy_batch_add(b, members.back()) == OSY_OK);
  }
  EXPECT(osy_batch_step(b, 3) == OSY_OK);
  EXPECT(fake::state().batch_launches == 3);
  EXPECT(fake::state().launches.empty());
  osy_batch_destroy(b);
  for (osy_fluid* fl : members) osy_fluid_destroy(fl);
}

// The starting shape follows the sweeps a call asks for, not only those the
// handle was made with; a chosen shape stays.
void project_shape_follows_sweeps() {
  osy_fluid *one = create(config(1920, 1080, 1)), *fifty = create(config(1920, 1080, 50));
  EXPECT(osy_fluid_project(one, 50, nullptr) == OSY_OK);
  EXPECT(osy_fluid_project(fifty, 50, nullptr) == OSY_OK);
  EXPECT(osy_fluid_synchronize(one) == OSY_OK);
  EXPECT(osy_fluid_synchronize(fifty) == OSY_OK);
  const auto& did = fake::state().launches;
  EXPECT(did.size() == 2 && did[0].tuning.k == did[1].tuning.k &&
         did[0].tuning.th == did[1].tuning.th);
  const osy_tuning chosen = shape(2, 8, 2);
  EXPECT(osy_fluid_set_tuning(one, &chosen) == OSY_OK);
  EXPECT(osy_fluid_project(one, 50, nullptr) == OSY_OK);
  EXPECT(osy_fluid_synchronize(one) == OSY_OK);
  EXPECT(did.back().tuning.k == 2);
  osy_fluid_destroy(one);
  osy_fluid_destroy(fifty);
}

// The launches a projection is said to make are those it makes: starting and
// chosen shapes, one launch or one per stage.
void launches_are_counted() {
  const osy_tuning starting = shape(-1, 0, 0);
  for (const osy_tuning& t : {starting, shape(2, 8, 2), shape(3, 12, 5), shape(3, 8, 4)}) {
    for (const float d_t : {0.05f, 2.0f}) {
      osy_config c = config(640, 480, 1, t.sweeps_per_launch != 5);  // (sums: up to 64 rows)
      c.d_t = d_t;
      osy_fluid* fl = create(c);
      if (t.projection_kernel >= 0) EXPECT(osy_fluid_set_tuning(fl, &t) == OSY_OK);
      for (const int sweeps : {0, 1, 7, 50}) {
        int32_t said = -1;
        EXPECT(osy_fluid_project_launches(fl, sweeps, &said) == OSY_OK);
        EXPECT(osy_fluid_project(fl, sweeps, nullptr) == OSY_OK);
        EXPECT(osy_fluid_synchronize(fl) == OSY_OK);
        if (sweeps == 0) {
          EXPECT(said == 0);
          continue;
        }
        const fake::Launch& did = fake::state().launches.back();
        const int k = did.tuning.k;
        EXPECT(did.sweeps == sweeps && said == (did.resident ? 1 : (sweeps + k - 1) / k));
      }
      osy_fluid_destroy(fl);
    }
  }
}

const std::map<std::string, void (*)()> kScenarios = {
    {"exchange_out_of_memory", exchange_out_of_memory},
    {"autotune_fails", autotune_fails},
    {"autotune_without_exchange", autotune_without_exchange},
    {"autotune_times_out", autotune_times_out},
    {"batch_autotune_times_out", batch_autotune_times_out},
    {"cleaned_in_stream_order", cleaned_in_stream_order},
    {"captured_projection", captured_projection},
    {"exchange_is_counted", exchange_is_counted},
    {"exchange_in_a_budget", exchange_in_a_budget},
    {"resident_says_what_runs", resident_says_what_runs},
    {"dividing_is_resident", dividing_is_resident},
    {"staging_is_bounded", staging_is_bounded},
    {"staging_shares_the_link", staging_shares_the_link},
    {"batch_division", batch_division},
    {"project_shape_follows_sweeps", project_shape_follows_sweeps},
    {"launches_are_counted", launches_are_counted},
};

}  // namespace

int main(int argc, char** argv) {
  if (argc != 2 || !kScenarios.count(argv[1])) {
    for (const auto& s : kScenarios) std::printf("%s\n", s.first.c_str());
    return 2;
  }
  kScenarios.at(argv[1])();
  for (const std::string& v : fake::state().violations) {
    std::printf("violation: %s\n", v.c_str());
    g_failed = 1;
  }
  if (!g_failed) std::printf("ok\n");
  return g_failed;
}
