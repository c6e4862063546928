// Host check of csrc/schedule.cpp and csrc/schedule_capture.cpp against a stand-in for the HIP runtime that keeps count: work counts as pending until
// finish() is called, and while a stream is being captured a call that asks or waits spoils the capture - from a thread that
// is not in the relaxed mode any such call, from a relaxed one a device-wide wait and anything that asks an event last
// recorded on that stream (as the runtime does on a gfx950 system).  Operators are stand-ins too.  No GPU.
#include <hip/hip_runtime.h>

#include <cstdio>
#include <cstdlib>
#include <map>
#include <new>
#include <set>
#include <utility>
#include <vector>

#include "common.h"
#include "d3d_spconv.h"

static bool noMemory = false;  // host allocations fail
void* operator new(size_t n) {
  void* p = noMemory ? nullptr : std::malloc(n);
  if (!p) throw std::bad_alloc();
  return p;
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, size_t) noexcept { std::free(p); }

namespace {
int pendingWork = 0, graphLaunches = 0, steps = 0, captures = 0, refusals = 0, liveGraphs = 0, liveEvents = 0, liveStreams = 0;
hipStream_t const kMain = reinterpret_cast<hipStream_t>(8), kOther = reinterpret_cast<hipStream_t>(12);
hipStream_t captured = nullptr;  // the stream that the caller captures
bool spoiled = false, destroyedRunning = false, refuseCapture = false, deviceWait = false;
hipStreamCaptureMode threadMode = hipStreamCaptureModeGlobal;
uint64_t operatorChanges = 0;
std::map<void*, bool> eventPending;
std::map<void*, hipStream_t> recordedOn;
std::set<void*> running;  // graphs launched and not finished
// the graph that the caller captures: its nodes with what each comes behind, and what the stream's next one will
bool capturing = false;
std::vector<std::pair<hipGraphNode_t, std::vector<hipGraphNode_t>>> nodes;
std::vector<hipGraphNode_t> behind;
int failAt = -1, emptyAt = -1;  // the step from now that fails / that enqueues nothing
uintptr_t nextHandle = 16;
void* fresh() { return reinterpret_cast<void*>(nextHandle += 16); }
hipError_t unsafe() {
  if (!captured || threadMode == hipStreamCaptureModeRelaxed) return hipSuccess;
  spoiled = true;
  return hipErrorStreamCaptureUnsupported;
}
void finish() {
  pendingWork = 0;
  running.clear();
  for (auto& e : eventPending) e.second = false;
}
}  // namespace

// ---- the runtime ----
extern "C" {
const char* hipGetErrorString(hipError_t) { return "stand-in error"; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode* m) {
  const hipStreamCaptureMode was = threadMode;
  threadMode = *m;
  *m = was;
  return hipSuccess;
}
hipError_t hipDeviceSynchronize() {
  deviceWait = true;
  if (captured) {
    spoiled = true;
    return hipErrorStreamCaptureUnsupported;
  }
  finish();
  return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
  *s = static_cast<hipStream_t>(fresh());
  ++liveStreams;
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) {
  --liveStreams;
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) {
  const hipError_t e = unsafe();
  if (e == hipSuccess) finish();
  return e;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
  *e = static_cast<hipEvent_t>(fresh());
  ++liveEvents;
  return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e) {
  eventPending.erase(e);
  --liveEvents;
  return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  eventPending[e] = pendingWork > 0;
  recordedOn[e] = s;
  return hipSuccess;
}
hipError_t unsafeFor(hipEvent_t e) {
  if (captured && recordedOn[e] == captured) {
    spoiled = true;
    return hipErrorCapturedEvent;
  }
  return unsafe();
}
hipError_t hipEventQuery(hipEvent_t e) {
  const hipError_t r = unsafeFor(e);
  return r != hipSuccess ? r : (eventPending[e] ? hipErrorNotReady : hipSuccess);
}
hipError_t hipEventSynchronize(hipEvent_t e) {
  const hipError_t r = unsafeFor(e);
  if (r == hipSuccess && eventPending[e]) finish();
  return r;
}
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t e, unsigned) {
  return captured && recordedOn[e] == captured ? hipErrorStreamCaptureIsolation : hipSuccess;
}
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus* st) {
  *st = hipStreamCaptureStatusNone;
  return hipSuccess;
}
hipError_t hipGraphCreate(hipGraph_t* g, unsigned) {
  *g = static_cast<hipGraph_t>(fresh());
  refusals += refuseCapture;
  return refuseCapture ? hipErrorStreamCaptureUnsupported : hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipStreamBeginCaptureToGraph(hipStream_t, hipGraph_t, const hipGraphNode_t*, const hipGraphEdgeData*, size_t,
                                        hipStreamCaptureMode) {
  return hipSuccess;
}
hipError_t hipStreamUpdateCaptureDependencies(hipStream_t s, hipGraphNode_t* deps, size_t n, unsigned flags) {
  if (s != kMain || !capturing || flags != hipStreamSetCaptureDependencies) return hipErrorIllegalState;
  behind.assign(deps, deps + n);
  return hipSuccess;
}
hipError_t hipStreamGetCaptureInfo_v2(hipStream_t s, hipStreamCaptureStatus* st, unsigned long long*, hipGraph_t*,
                                      const hipGraphNode_t** deps, size_t* n) {
  if (s == kMain) {
    *st = capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
    *deps = behind.data();
    *n = behind.size();
    return hipSuccess;
  }
  *st = hipStreamCaptureStatusActive;
  *deps = nullptr;
  *n = 0;
  return hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t*) { return hipSuccess; }
hipError_t hipGraphInstantiateWithFlags(hipGraphExec_t* g, hipGraph_t, unsigned long long) {
  *g = static_cast<hipGraphExec_t>(fresh());
  ++captures;
  ++liveGraphs;
  return hipSuccess;
}
hipError_t hipGraphExecDestroy(hipGraphExec_t g) {
  if (running.count(g)) destroyedRunning = true;
  --liveGraphs;
  return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t g, hipStream_t) {
  ++graphLaunches;
  ++pendingWork;
  running.insert(g);
  return hipSuccess;
}
// ---- the operators ----
const char* d3d_plugin_type(const d3d_plugin*) { return "BEVDensify"; }
int32_t d3d_num_outputs(const d3d_plugin*) { return 1; }
int32_t d3d_enqueue(d3d_plugin*, const d3d_tensor_desc*, const d3d_tensor_desc*, const void* const*, void* const*, void*, size_t,
                    void* stream) {
  if (failAt >= 0 && failAt-- == 0) return D3D_ERR_UNSUPPORTED;
  ++steps;
  if (capturing && stream == kMain) {
    if (emptyAt >= 0 && emptyAt-- == 0) return D3D_OK;
    const auto node = static_cast<hipGraphNode_t>(fresh());
    nodes.emplace_back(node, behind);
    behind = {node};
    return D3D_OK;
  }
  ++pendingWork;
  return D3D_OK;
}
}
namespace d3d {
void setError(const char*, ...) {}
uint64_t pluginChanges(const d3d_plugin*) { return operatorChanges; }
int32_t launchSum(int32_t, const void*, const void*, void*, int64_t, hipStream_t) { return D3D_OK; }
int32_t launchCastFromFloat(int32_t, const float*, void*, int64_t, hipStream_t) { return D3D_OK; }
}  // namespace d3d

#define CHECK(cond)                                                                \
  do {                                                                             \
    if (!(cond)) {                                                                 \
      std::fprintf(stderr, "schedule_check: %s failed (line %d)\n", #cond, __LINE__); \
      return 1;                                                                    \
    }                                                                              \
  } while (0)

namespace {
d3d_schedule* make() {
  d3d_schedule* s = nullptr;
  if (d3d_schedule_create(2, &s) != D3D_OK) return nullptr;
  static d3d_tensor_desc in[4], out[1];
  const void* ins[4] = {};
  void* outs[1] = {};
  auto* op = reinterpret_cast<d3d_plugin*>(16);
  const int32_t first = d3d_schedule_add(s, op, in, 4, out, 1, ins, outs, nullptr, 0, 1, nullptr, 0);
  d3d_schedule_add(s, op, in, 4, out, 1, ins, outs, nullptr, 0, 0, &first, 1);
  return s;
}

// A schedule destroyed while the caller captures a stream, its last launch still running.
int destroyUnderCapture() {
  for (hipStream_t during : {kOther, kMain}) {
    d3d_schedule* s = make();
    const int launched = graphLaunches;
    for (int i = 0; i < 5; ++i) CHECK(d3d_schedule_run(s, kMain) == D3D_OK);
    CHECK(graphLaunches == launched + 3 && liveGraphs == 1);
    captured = during;
    d3d_schedule_destroy(s);
    CHECK(!spoiled && !destroyedRunning && !deviceWait && threadMode == hipStreamCaptureModeGlobal);
    CHECK(liveGraphs == (during == kMain ? 1 : 0));
    captured = nullptr;
    finish();
    d3d_schedule_destroy(make());
    CHECK(liveGraphs == 0 && liveStreams == 0 && liveEvents == 0 && !destroyedRunning);
  }
  return 0;
}

// A change under a graph whose launch still runs: the run neither waits nor destroys it; it goes once it has run.
int changeWithoutWaiting() {
  d3d_schedule* s = make();
  for (int i = 0; i < 5; ++i) CHECK(d3d_schedule_run(s, kMain) == D3D_OK);
  const int launched = graphLaunches, before = captures;
  ++operatorChanges;
  captured = kOther;
  for (int i = 0; i < 4; ++i) CHECK(d3d_schedule_run(s, kMain) == D3D_OK);
  CHECK(graphLaunches == launched + 2 && captures == before + 1);
  CHECK(!spoiled && !destroyedRunning && !deviceWait && pendingWork > 0 && liveGraphs == 2);
  captured = nullptr;
  finish();
  CHECK(d3d_schedule_run(s, kMain) == D3D_OK && liveGraphs == 1);
  d3d_schedule_destroy(s);
  CHECK(liveGraphs == 0 && liveStreams == 0 && liveEvents == 0 && !destroyedRunning);
  return 0;
}

// A capture that is refused for a while: the passes run step by step, the attempts get rarer, and the graph comes in the end.
int refusedForAWhile() {
  d3d_schedule* s = make();
  refuseCapture = true;
  const int launched = graphLaunches;
  refusals = 0;
  for (int i = 0; i < 40; ++i) CHECK(d3d_schedule_run(s, kMain) == D3D_OK);
  CHECK(graphLaunches == launched && refusals >= 3 && refusals <= 5);
  refuseCapture = false;
  for (int i = 0; i < 100; ++i) CHECK(d3d_schedule_run(s, kMain) == D3D_OK);
  CHECK(graphLaunches > launched);
  ++operatorChanges;  // the next graph comes as fast as the first one
  const int before = graphLaunches;
  for (int i = 0; i < 3; ++i) CHECK(d3d_schedule_run(s, kMain) == D3D_OK);
  CHECK(graphLaunches == before + 1);
  d3d_schedule_destroy(s);
  return 0;
}

// Host memory that runs out is a status, not an exception in the caller's language.
int outOfHostMemory() {
  d3d_schedule *s = make(), *none = nullptr;
  const int32_t size = d3d_schedule_size(s);
  d3d_tensor_desc in[4], out[1];
  const void* ins[4] = {};
  void* outs[1] = {};
  noMemory = true;
  const int32_t created = d3d_schedule_create(1, &none);
  const int32_t added = d3d_schedule_add(s, reinterpret_cast<d3d_plugin*>(16), in, 4, out, 1, ins, outs, nullptr, 0, 0, nullptr, 0);
  const int32_t summed = d3d_schedule_add_sum(s, D3D_FLOAT, in, in, in, 1, 0, nullptr, 0);
  noMemory = false;
  CHECK(created < 0 && !none && added < 0 && summed < 0 && d3d_schedule_size(s) == size);
  CHECK(d3d_schedule_run(s, kMain) == D3D_OK);
  d3d_schedule_destroy(s);
  return 0;
}

// A pass of five steps: two rulebooks on lanes of their own, the second behind the first, three convolutions on lane 0, each
// behind its rulebook (the third behind the second's again).
d3d_schedule* pass() {
  d3d_schedule* s = nullptr;
  if (d3d_schedule_create(3, &s) != D3D_OK) return nullptr;
  static d3d_tensor_desc in[4], out[1];
  const void* ins[4] = {};
  void* outs[1] = {};
  auto* op = reinterpret_cast<d3d_plugin*>(16);
  auto add = [&](int32_t lane, std::initializer_list<int32_t> after) {
    return d3d_schedule_add(s, op, in, 4, out, 1, ins, outs, nullptr, 0, lane, after.begin(), static_cast<int32_t>(after.size()));
  };
  const int32_t r1 = add(1, {}), c1 = add(0, {r1}), r2 = add(2, {r1}), c2 = add(0, {r2});
  add(0, {r2, c2});
  (void)c1;
  return s;
}

void beginCapture(std::vector<hipGraphNode_t> base) {
  capturing = true;
  captured = kMain;
  nodes.clear();
  behind = std::move(base);
}
void endCapture() {
  capturing = false;
  captured = nullptr;
  failAt = emptyAt = -1;
}
const std::vector<hipGraphNode_t>& behindNode(size_t i) { return nodes[i].second; }
std::vector<hipGraphNode_t> named(std::initializer_list<size_t> which) {
  std::vector<hipGraphNode_t> v;
  for (size_t i : which) v.push_back(nodes[i].first);
  return v;
}

// The steps as nodes of the caller's graph: behind what the stream held or behind the steps they wait for, without edges that others
// imply, the stream going on behind all of them; no stream and no event is made, and none is touched.
int captureOfSteps() {
  auto* const held = static_cast<hipGraphNode_t>(fresh());
  auto* const held2 = static_cast<hipGraphNode_t>(fresh());
  d3d_schedule* s = pass();
  CHECK(s && d3d_schedule_size(s) == 5 && liveStreams == 0 && liveEvents == 0);
  CHECK(d3d_schedule_capture(s, kMain) == D3D_ERR_UNSUPPORTED && steps >= 0);  // not capturing: nothing enqueued
  const int before = steps;
  beginCapture({held, held2});
  CHECK(d3d_schedule_capture(s, kMain) == D3D_OK);
  CHECK(steps == before + 5 && nodes.size() == 5 && liveStreams == 0 && liveEvents == 0 && !spoiled);
  CHECK((behindNode(0) == std::vector<hipGraphNode_t>{held, held2}));
  CHECK(behindNode(1) == named({0}) && behindNode(2) == named({0}));
  CHECK(behindNode(3) == named({1, 2}) && behindNode(4) == named({3}) && behind == named({4}));
  CHECK(d3d_schedule_run(s, kOther) == D3D_OK);  // the same schedule eagerly, while kMain is captured
  CHECK(liveStreams == 2 && liveEvents > 0 && !spoiled && nodes.size() == 5);
  CHECK(d3d_schedule_capture(s, kMain) == D3D_OK && nodes.size() == 10);  // and a second time into the same graph
  CHECK(behindNode(5) == named({4}) && behind == named({9}));
  endCapture();
  finish();
  d3d_schedule_destroy(s);
  CHECK(liveStreams == 0 && liveEvents == 0);
  return 0;
}

// A step that fails ends the capture's steps: an error, never the status that says nothing was captured, and the stream goes on
// behind what was.  A step that enqueues nothing stands for what it came behind.
int captureOfFailingAndEmptySteps() {
  auto* const held = static_cast<hipGraphNode_t>(fresh());
  for (int at = 0; at < 5; ++at) {
    d3d_schedule* s = pass();
    beginCapture({held});
    failAt = at;
    const int32_t rc = d3d_schedule_capture(s, kMain);
    CHECK(rc < 0 && rc != D3D_ERR_UNSUPPORTED && nodes.size() == static_cast<size_t>(at));
    if (at == 0) CHECK(behind == std::vector<hipGraphNode_t>{held});
    if (at == 1) CHECK(behind == named({0}));
    if (at == 2) CHECK(behind == named({1, 0}));
    if (at == 3) CHECK(behind == named({1, 2}));
    if (at == 4) CHECK(behind == named({3}));
    endCapture();
    d3d_schedule_destroy(s);
  }
  d3d_schedule* s = pass();
  beginCapture({held});
  emptyAt = 0;  // the first rulebook
  CHECK(d3d_schedule_capture(s, kMain) == D3D_OK && nodes.size() == 4);
  CHECK((behindNode(0) == std::vector<hipGraphNode_t>{held}) && (behindNode(1) == std::vector<hipGraphNode_t>{held}));
  CHECK(behindNode(2) == named({0, 1}) && behind == named({3}));
  beginCapture({});  // a stream that holds nothing yet
  emptyAt = 2;       // the second rulebook: the convolutions behind it come behind what it did
  CHECK(d3d_schedule_capture(s, kMain) == D3D_OK && nodes.size() == 4);
  CHECK(behindNode(0).empty() && behindNode(2) == named({1, 0}) && behind == named({3}));
  endCapture();
  d3d_schedule* none = nullptr;
  CHECK(d3d_schedule_create(1, &none) == D3D_OK);
  beginCapture({held});
  CHECK(d3d_schedule_capture(none, kMain) == D3D_OK && (behind == std::vector<hipGraphNode_t>{held}));  // no steps
  endCapture();
  d3d_schedule_destroy(none);
  d3d_schedule_destroy(s);
  CHECK(liveStreams == 0 && liveEvents == 0);
  return 0;
}
}  // namespace

int main() {
  if (captureOfSteps() || captureOfFailingAndEmptySteps()) return 1;
  if (destroyUnderCapture() || changeWithoutWaiting() || refusedForAWhile() || outOfHostMemory()) return 1;
  std::puts("schedule_check ok");
  return 0;
}
