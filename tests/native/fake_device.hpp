// The host runtime's device, played on the host: the HIP calls and kernel launches that engine.cpp
// makes, with a stream that runs nothing before somebody waits for it (the host gets as far ahead
// of the device as it may). Kernels do what the host sees of them, the epilogues' hours, rows and
// states; agents stay where they are. A test scripts the device's events in `fake`.
#pragma once
#include <hip/hip_runtime_api.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <deque>
#include <functional>
#include <string>
#include <vector>

#include "epirust_gpu.h"
#include "init.hpp"
#include "kernels.hpp"
#include "stream.hpp"

struct Fake {
  uint32_t stop_hour = ~0u;  // nobody is ill any more from this hour on
  uint32_t lock_hour = ~0u;  // a lockdown comes at this hour
  uint32_t exposed_until = 0;  // the last hour after which somebody is exposed
  bool maps_fail = false;    // building the office layout's slot maps fails
  int copies_before_failure = -1;  // of tables to the device, while it is not negative
  bool wrong_blocks = false;  // a launch whose threads per block are not its table's
  uint32_t captures = 0, graphs = 0;  // graphs instantiated, and launched
  std::vector<std::string> launches;  // kernels run, the idle ones of stopped runs as "idle"
  uint32_t count(const std::string& name) const {
    uint32_t n = 0;
    for (const std::string& s : launches) n += s == name;
    return n;
  }
};
inline Fake fake;

using Work = std::function<void()>;
struct FakeGraph {
  std::vector<Work> nodes;
};
inline std::deque<Work> fake_stream;
inline FakeGraph* fake_capture = nullptr;
inline void enqueue(Work w) {
  if (fake_capture) fake_capture->nodes.push_back(std::move(w));
  else fake_stream.push_back(std::move(w));
}
inline void drain() {
  while (!fake_stream.empty()) {
    Work w = std::move(fake_stream.front());
    fake_stream.pop_front();
    w();
  }
}
struct FakeEvent {
  uint64_t recorded = 0, passed = 0;
};

extern "C" {
hipError_t hipGetDeviceCount(int* n) { return *n = 1, hipSuccess; }
hipError_t hipGetDevice(int* d) { return *d = 0, hipSuccess; }
hipError_t hipGetDeviceProperties(hipDeviceProp_t* p, int) {
  std::memset(p, 0, sizeof *p);
  std::strcpy(p->gcnArchName, "gfx950");
  return hipSuccess;
}
const char* hipGetErrorString(hipError_t) { return "fake error"; }
hipError_t hipMalloc(void** p, size_t n) { return *p = std::calloc(n, 1), hipSuccess; }
hipError_t hipFree(void* p) { return std::free(p), hipSuccess; }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { return *p = std::calloc(n, 1), hipSuccess; }
hipError_t hipHostFree(void* p) { return std::free(p), hipSuccess; }
hipError_t hipHostGetDevicePointer(void** d, void* h, unsigned) { return *d = h, hipSuccess; }
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) { return std::memcpy(d, s, n), hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
  if (fake.copies_before_failure >= 0 && fake.copies_before_failure-- == 0) return hipErrorUnknown;
  enqueue([=] { std::memcpy(d, s, n); });
  return hipSuccess;
}
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) {
  enqueue([=] { std::memset(d, v, n); });
  return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { return *s = nullptr, hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return drain(), hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return drain(), hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) {
  fake_capture = new FakeGraph;
  return hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) {
  *g = reinterpret_cast<hipGraph_t>(fake_capture);
  fake_capture = nullptr;
  return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t g, hipGraphNode_t*, char*, size_t) {
  ++fake.captures;
  *e = reinterpret_cast<hipGraphExec_t>(new FakeGraph(*reinterpret_cast<FakeGraph*>(g)));
  return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t g) { return delete reinterpret_cast<FakeGraph*>(g), hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t e) { return delete reinterpret_cast<FakeGraph*>(e), hipSuccess; }
hipError_t hipGraphLaunch(hipGraphExec_t e, hipStream_t) {
  ++fake.graphs;
  for (const Work& w : reinterpret_cast<FakeGraph*>(e)->nodes) enqueue(w);
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
  *e = reinterpret_cast<hipEvent_t>(new FakeEvent);
  return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t* e) { return hipEventCreateWithFlags(e, 0); }
hipError_t hipEventDestroy(hipEvent_t e) { return delete reinterpret_cast<FakeEvent*>(e), hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t) {
  FakeEvent* f = reinterpret_cast<FakeEvent*>(e);
  const uint64_t k = ++f->recorded;
  enqueue([f, k] { f->passed = k; });
  return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) {  // runs no further than the event
  FakeEvent* f = reinterpret_cast<FakeEvent*>(e);
  while (f->passed < f->recorded && !fake_stream.empty()) {
    Work w = std::move(fake_stream.front());
    fake_stream.pop_front();
    w();
  }
  return hipSuccess;
}
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { return *ms = 0.0f, hipSuccess; }
}

namespace epi {

// The epilogues of `hours` hours, from the simulations' states on.
inline void fake_epilogues(const DevView& v, const LaunchShape& s, uint32_t hours) {
  for (uint32_t i = 0; i < s.n_sims; ++i) {
    SimState& st = v.state[i];
    const SimDesc& D = v.desc[i];
    for (uint32_t k = 0; k < hours && st.active; ++k) {
      const uint32_t h = ++st.hour;
      st.rows_written = h;
      v.rows[D.row_off + h - 1] = v.host_rows[D.row_off + h - 1] = Counts7{h, D.n, 0, 0, 0, 0, 0};
      st.last_counts[1] = h <= fake.exposed_until;
      if (h == fake.lock_hour) st.locked = 1;
      if (h >= fake.stop_hour || h + 1 >= D.hours) st.active = 0;
      v.host_state[i] = st;
    }
  }
}
inline bool running(const DevView& v, const LaunchShape& s) {
  for (uint32_t i = 0; i < s.n_sims; ++i)
    if (v.state[i].active) return true;
  return false;
}
// A launch over the agents: every block but a simulation's last (or, of offices, any) is full, so
// more or fewer threads than the table was built for repeat agents or leave some out.
inline void over_agents(const char* name, const DevView& v, const LaunchShape& s, std::function<void()> then = {}) {
  enqueue([=] {
    fake.launches.push_back(running(v, s) ? name : "idle");
    const uint32_t blocks = v.office ? s.office_agent_blocks : s.agent_blocks;
    const uint32_t threads = v.office ? s.office_block : s.block;
    std::vector<uint64_t> agents(s.n_sims, 0);
    for (uint32_t b = 0; b < blocks; ++b) {
      const AgentBlock& e = v.agent_blocks[b];
      agents[e.sim] += e.count;
      if (e.count > threads) fake.wrong_blocks = true;
      if (!v.office && e.count != threads && e.first + e.count != v.desc[e.sim].n) fake.wrong_blocks = true;
    }
    for (uint32_t i = 0; i < s.n_sims; ++i)
      if (agents[i] != v.desc[i].n) fake.wrong_blocks = true;
    if (then) then();
  });
}

hipError_t launch_hospital_scan(const DevView& v, const LaunchShape& s, hipStream_t) {
  enqueue([=] { fake.launches.push_back(running(v, s) ? "scan" : "idle"); });
  return hipSuccess;
}
hipError_t launch_step(const DevView& v, const LaunchShape& s, uint32_t, hipStream_t) {
  return over_agents("step", v, s), hipSuccess;
}
hipError_t launch_commit(const DevView& v, const LaunchShape& s, uint32_t, hipStream_t) {
  return over_agents("commit", v, s, [=] { fake_epilogues(v, s, 1); }), hipSuccess;
}
hipError_t launch_rest(const DevView& v, const LaunchShape& s, uint32_t, hipStream_t) {
  return over_agents("rest", v, s, [=] { fake_epilogues(v, s, 1); }), hipSuccess;
}
hipError_t launch_night(const DevView& v, const LaunchShape& s, hipStream_t) {
  return over_agents("night", v, s, [=] { fake_epilogues(v, s, 6); }), hipSuccess;
}
hipError_t launch_quiet_hours(const DevView& v, const LaunchShape& s, uint32_t n_hours, hipStream_t) {
  enqueue([=] {
    fake.launches.push_back(running(v, s) ? "quiet" : "idle");
    fake_epilogues(v, s, n_hours);
  });
  return hipSuccess;
}
hipError_t launch_relayout(const DevView& home, const DevView&, const TileRef*, uint32_t, bool, hipStream_t) {
  enqueue([=] { fake.launches.push_back("relayout"); });
  return hipSuccess;
}
hipError_t launch_apply_sweep(const DevView& v, const LaunchShape& s, hipStream_t) {
  return over_agents("sweep", v, s), hipSuccess;
}
hipError_t launch_fill_u32(uint32_t* p, uint64_t n, uint32_t value, hipStream_t) {
  enqueue([=] { std::fill_n(p, n, value); });
  return hipSuccess;
}
hipError_t launch_export_active(const DevView& v, uint32_t n_sims, uint32_t* active, hipStream_t) {
  enqueue([=] {
    for (uint32_t i = 0; i < n_sims; ++i) active[i] = v.state[i].active;
  });
  return hipSuccess;
}
hipError_t launch_citizen_states(const StreamArgs&, hipStream_t) { return hipErrorUnknown; }
hipError_t noalloc_scratch(unsigned long long** p) { return *p = nullptr, hipSuccess; }
uint32_t max_record_bytes(uint32_t, uint32_t, uint32_t) { return kMaxRecord; }
uint32_t stream_blocks(uint32_t n) { return (n + 255) / 256; }

hipError_t synthesize_on_device(const std::vector<InitJob>&, hipStream_t, std::string&) { return hipSuccess; }
// Every agent works, in office id % n_offices.
hipError_t build_office_maps_on_device(const std::vector<OfficeJob>& jobs,
                                       std::vector<std::vector<uint32_t>>& workers_per_office, hipStream_t,
                                       std::string& err) {
  if (fake.maps_fail) return err = "fake", hipErrorOutOfMemory;
  workers_per_office.assign(jobs.size(), {});
  for (size_t i = 0; i < jobs.size(); ++i) {
    workers_per_office[i].assign(jobs[i].n_offices, 0);
    for (uint32_t id = 0; id < jobs[i].n; ++id) ++workers_per_office[i][id % jobs[i].n_offices];
  }
  return hipSuccess;
}

}  // namespace epi
