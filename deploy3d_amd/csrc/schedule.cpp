// A schedule: a recorded sequence of operator enqueues, replayed from native code on several HIP streams or as one HIP graph.
//
// What TensorRT's execution context does for the reference (IExecutionContext::enqueueV3 walking the engine's
// layers; deploy3d/symfun/trt_utils/trt_onnx_module.py:186-250 drives it): the caller describes a pass once -
// operator, descriptors, device pointers, workspace per step, the lane (stream) it runs on and the earlier
// steps it has to wait for - and `d3d_schedule_run` then enqueues the whole pass without going back to the
// caller's language between operators.  Lane 0 is the stream passed to run; the other lanes are streams the
// schedule owns.  Steps of one lane run in the order they were added; a step waits for the steps named in `after`
// through events, recorded only behind steps that somebody on another lane waits for.  All lanes fork from
// lane 0 when a run starts and join it when the run ends, so for the caller a run is ordinary stream-ordered work
// on its stream.
//
// From the third run on the pass is one HIP graph: every step is captured into it behind the nodes of the steps it
// waits for (explicit dependencies, no cross-stream events), and a run is one graph launch.  A pass of a small scan (36
// launches, 9 000 voxels) costs the host 415 us step by step on three lanes - more than its kernels take - and 195 as a
// graph; the device then takes 345 us.  The graph is dropped when an operator reports a change (pluginChanges).
//
// A dropped graph is destroyed once its last launch has run (RetiredGraph): no device-wide synchronisation, which a stream
// under capture would not survive, and no event behind every launch, which costs 4 to 6 us a pass.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstring>
#include <memory>
#include <mutex>
#include <utility>

#include "schedule.h"

namespace d3d {

int32_t scheduleEnqueueStep(const d3d_schedule::Step& st, hipStream_t q) {
  switch (st.kind) {
    case d3d_schedule::kSum: return d3d::launchSum(st.dtype, st.inputs[0], st.inputs[1], st.outputs[0], st.count, q);
    case d3d_schedule::kCast:
      return d3d::launchCastFromFloat(st.dtype, static_cast<const float*>(st.inputs[0]), st.outputs[0], st.count, q);
    default:
      return d3d_enqueue(st.plugin, st.in.data(), st.out.data(), st.inputs.data(), st.outputs.data(), st.workspace,
                         st.workspaceBytes, q);
  }
}

// A dependency that another one implies gets no edge: every edge between branches is a wait packet in front of the kernel, 6 us
// even when the other branch is long done (a VoxelNet backbone of 9 000 voxels: 374 us with the implied edges, 324 without;
// 120 000 voxels: 708 and 700).
std::vector<std::vector<int>> scheduleEdges(const d3d_schedule* s) {
  const size_t count = s->steps.size();
  std::vector<std::vector<int>> edges(count);
  std::vector<std::vector<bool>> behindOf(count, std::vector<bool>(count));  // what each step comes after, directly or not
  for (size_t i = 0; i < count; ++i) {
    const d3d_schedule::Step& st = s->steps[i];
    std::vector<int> direct(st.after);
    if (st.before >= 0) direct.insert(direct.begin(), st.before);
    for (int d : direct) {
      behindOf[i][static_cast<size_t>(d)] = true;
      for (size_t k = 0; k < count; ++k)
        if (behindOf[static_cast<size_t>(d)][k]) behindOf[i][k] = true;
    }
    auto implied = [&](int d) {
      for (int other : direct)
        if (behindOf[static_cast<size_t>(other)][static_cast<size_t>(d)]) return true;
      return false;
    };
    for (int d : direct)
      if (!implied(d)) edges[i].push_back(d);
  }
  return edges;
}

}  // namespace d3d

namespace {

int32_t hipFail(hipError_t e, const char* what) {
  d3d::setError("schedule: %s failed: %s", what, hipGetErrorString(e));
  return D3D_ERR_DEVICE;
}

uint64_t changesOf(const d3d_schedule* s) {
  uint64_t sum = 0;
  for (const auto& st : s->steps)
    if (st.plugin) sum += d3d::pluginChanges(st.plugin);
  return sum;
}

// Asking an event or waiting for one is legal while another stream is being captured in the global mode only from a thread in
// the relaxed mode; from any other it fails and spoils that capture.
struct RelaxedCapture {
  hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
  RelaxedCapture() { (void)hipThreadExchangeStreamCaptureMode(&mode); }
  ~RelaxedCapture() { (void)hipThreadExchangeStreamCaptureMode(&mode); }
};

// A graph that no schedule launches any more, until its last launch has run.  What tells is an event (`over`) on a stream of
// its own (`behind`) that waits for an event (`ran`) on the stream of the launch.  The latter itself may not be asked: if
// that stream is being captured by then, even a relaxed query of an event last recorded on it spoils the capture.
struct RetiredGraph {
  hipGraphExec_t graph = nullptr;
  hipStream_t launchedOn = nullptr;  // until `ran` has been recorded there
  hipEvent_t ran = nullptr, over = nullptr;
  hipStream_t behind = nullptr;
  bool marked = false;
};

// Puts `over` behind the graph's last launch; false while the stream of the launch is being captured.
bool mark(RetiredGraph& g) {
  if (g.marked) return true;
  hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(g.launchedOn, &capture) != hipSuccess || capture != hipStreamCaptureStatusNone) return false;
  if (!g.ran && hipEventCreateWithFlags(&g.ran, hipEventDisableTiming) != hipSuccess) return false;
  if (!g.over && hipEventCreateWithFlags(&g.over, hipEventDisableTiming) != hipSuccess) return false;
  if (!g.behind && hipStreamCreateWithFlags(&g.behind, hipStreamNonBlocking) != hipSuccess) return false;
  g.marked = hipEventRecord(g.ran, g.launchedOn) == hipSuccess && hipStreamWaitEvent(g.behind, g.ran, 0) == hipSuccess &&
             hipEventRecord(g.over, g.behind) == hipSuccess;
  return g.marked;
}

struct Retired {
  std::mutex mutex;
  std::atomic<size_t> count{0};
  std::vector<RetiredGraph> graphs;
};
Retired& retired() {
  static Retired* r = new Retired();  // lives until the process ends
  return *r;
}

// Destroys the retired graphs that have run; `wait`: waits for each that can be waited for.
void reapGraphs(bool wait) {
  Retired& r = retired();
  if (r.count.load(std::memory_order_relaxed) == 0) return;
  const RelaxedCapture relaxed;
  std::lock_guard<std::mutex> lock(r.mutex);
  for (size_t i = 0; i < r.graphs.size();) {
    RetiredGraph& g = r.graphs[i];
    if (!mark(g) || (wait ? hipEventSynchronize(g.over) : hipEventQuery(g.over)) != hipSuccess) {
      (void)hipGetLastError();  // not ready, or not now: no error of the caller's
      ++i;
      continue;
    }
    (void)hipGraphExecDestroy(g.graph);
    (void)hipEventDestroy(g.ran);
    (void)hipEventDestroy(g.over);
    (void)hipStreamDestroy(g.behind);
    g = r.graphs.back();
    r.graphs.pop_back();
  }
  r.count.store(r.graphs.size(), std::memory_order_relaxed);
}

// `stream`: the stream of the last launch or one that the caller has ordered behind it.
void dropGraph(d3d_schedule* s, hipStream_t stream) {
  if (!s->graph) return;
  const RelaxedCapture relaxed;
  RetiredGraph g;
  g.graph = s->graph;
  g.launchedOn = stream;
  s->graph = nullptr;
  if (!s->launched) {
    (void)hipGraphExecDestroy(g.graph);
    return;
  }
  s->launched = false;
  if (!mark(g)) (void)hipGetLastError();
  Retired& r = retired();
  std::lock_guard<std::mutex> lock(r.mutex);
  r.graphs.push_back(g);
  r.count.store(r.graphs.size(), std::memory_order_relaxed);
}

// Captures every step into one graph, each behind the last nodes of the steps it waits for.  False (and no graph) if
// any part of it is refused; nothing has been enqueued then.
bool captureGraph(d3d_schedule* s) {
  hipGraph_t graph = nullptr;
  hipStream_t q = nullptr;
  bool ok;
  {
    const RelaxedCapture relaxed;
    if (hipGraphCreate(&graph, 0) != hipSuccess) {
      (void)hipGetLastError();
      return false;
    }
    ok = hipStreamCreateWithFlags(&q, hipStreamNonBlocking) == hipSuccess;
  }
  const size_t count = s->steps.size();
  std::vector<std::vector<hipGraphNode_t>> tail(count);
  const std::vector<std::vector<int>> edges = d3d::scheduleEdges(s);
  for (size_t i = 0; ok && i < count; ++i) {
    const d3d_schedule::Step& st = s->steps[i];
    std::vector<hipGraphNode_t> deps;
    for (int d : edges[i])
      for (hipGraphNode_t n : tail[static_cast<size_t>(d)])
        if (std::find(deps.begin(), deps.end(), n) == deps.end()) deps.push_back(n);
    if (hipStreamBeginCaptureToGraph(q, graph, deps.empty() ? nullptr : deps.data(), nullptr, deps.size(),
                                     hipStreamCaptureModeThreadLocal) != hipSuccess) {
      ok = false;
      break;
    }
    ok = d3d::scheduleEnqueueStep(st, q) == D3D_OK;
    hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
    const hipGraphNode_t* last = nullptr;
    size_t nLast = 0;
    if (ok) ok = hipStreamGetCaptureInfo_v2(q, &status, nullptr, nullptr, &last, &nLast) == hipSuccess;
    if (ok) tail[i].assign(last, last + nLast);
    hipGraph_t same = nullptr;
    ok = hipStreamEndCapture(q, &same) == hipSuccess && ok;
  }
  const RelaxedCapture relaxed;
  if (ok) ok = hipGraphInstantiateWithFlags(&s->graph, graph, 0) == hipSuccess;
  if (!ok) {
    s->graph = nullptr;
    (void)hipGetLastError();
  }
  (void)hipGraphDestroy(graph);
  if (q) (void)hipStreamDestroy(q);
  return ok;
}

// The streams and events of a run that enqueues step by step.
hipError_t makeLanes(d3d_schedule* s) {
  const RelaxedCapture relaxed;  // (a stream of the caller's may be capturing)
  hipError_t e = hipSuccess;
  auto event = [&](hipEvent_t& ev) {
    if (!ev && e == hipSuccess) e = hipEventCreateWithFlags(&ev, hipEventDisableTiming);
  };
  if (s->lanes.size() > 1) event(s->fork);
  for (size_t l = 1; l < s->lanes.size(); ++l) {
    if (!s->lanes[l] && e == hipSuccess) e = hipStreamCreateWithFlags(&s->lanes[l], hipStreamNonBlocking);  // default priority
    event(s->joined[l]);
  }
  for (auto& st : s->steps)
    if (st.awaited) event(st.done);
  return e;
}

// The checks and lane bookkeeping that every kind of step shares; returns the step's index or a status.
int32_t appendStep(d3d_schedule* s, d3d_schedule::Step&& st, const int32_t* after, int32_t nb_after) {
  const int me = static_cast<int>(s->steps.size());
  if (nb_after < 0 || (nb_after && !after) || st.lane < 0 || st.lane >= static_cast<int32_t>(s->lanes.size())) {
    d3d::setError("schedule: bad step (null array, negative count or lane outside the schedule)");
    return D3D_ERR_BAD_ARG;
  }
  for (int32_t i = 0; i < nb_after; ++i)
    if (after[i] < 0 || after[i] >= me) {
      d3d::setError("schedule: step %d waits for step %d, which does not precede it", me, after[i]);
      return D3D_ERR_BAD_ARG;
    }
  for (int32_t i = 0; i < nb_after; ++i) {
    d3d_schedule::Step& dep = s->steps[static_cast<size_t>(after[i])];
    if (dep.lane == st.lane) continue;  // stream order already holds
    dep.awaited = true;
    st.after.push_back(after[i]);
  }
  for (int i = me - 1; i >= 0 && st.before < 0; --i)
    if (s->steps[static_cast<size_t>(i)].lane == st.lane) st.before = i;
  dropGraph(s, s->launchedOn);
  s->lastChanges = ~0ull;
  s->steps.push_back(std::move(st));
  return me;
}

}  // namespace

extern "C" {

int32_t d3d_schedule_create(int32_t n_lanes, d3d_schedule** out) {
  D3D_GUARD_BEGIN
  if (!out || n_lanes < 1 || n_lanes > 8) {
    d3d::setError("schedule: 1 to 8 lanes");
    return D3D_ERR_BAD_ARG;
  }
  *out = nullptr;
  reapGraphs(false);
  auto s = std::make_unique<d3d_schedule>();
  s->lanes.assign(static_cast<size_t>(n_lanes), nullptr);
  s->joined.assign(static_cast<size_t>(n_lanes), nullptr);
  *out = s.release();
  return D3D_OK;
  D3D_GUARD_END(D3D_ERR_BAD_ARG)
}

void d3d_schedule_destroy(d3d_schedule* s) {
  D3D_GUARD_BEGIN
  if (!s) return;
  if (s->graph || s->lanes.size() > 1) {
    const RelaxedCapture relaxed;
    dropGraph(s, s->launchedOn);
    reapGraphs(true);
    for (auto& st : s->steps)
      if (st.done) (void)hipEventDestroy(st.done);
    for (size_t l = 1; l < s->lanes.size(); ++l) {
      if (s->joined[l]) {  // behind the lane's work of every run
        (void)hipEventSynchronize(s->joined[l]);
        (void)hipEventDestroy(s->joined[l]);
      }
      if (s->lanes[l]) (void)hipStreamDestroy(s->lanes[l]);
    }
    if (s->fork) (void)hipEventDestroy(s->fork);
  }
  delete s;
  D3D_GUARD_END()
}

int32_t d3d_schedule_add(d3d_schedule* s, d3d_plugin* plugin, const d3d_tensor_desc* in_desc, int32_t nb_in,
                         const d3d_tensor_desc* out_desc, int32_t nb_out, const void* const* inputs,
                         void* const* outputs, void* workspace, size_t workspace_bytes, int32_t lane,
                         const int32_t* after, int32_t nb_after) {
  D3D_GUARD_BEGIN
  if (!s || !plugin || nb_in < 0 || nb_out < 0 || nb_after < 0 || (nb_in && (!in_desc || !inputs)) ||
      (nb_out && (!out_desc || !outputs)) || (nb_after && !after) || lane < 0 ||
      lane >= static_cast<int32_t>(s->lanes.size())) {
    d3d::setError("schedule: bad step (null array, negative count or lane outside the schedule)");
    return D3D_ERR_BAD_ARG;
  }
  {
    // the operators read fixed positions of the input arrays: a shorter array is a host out-of-bounds read
    const char* type = d3d_plugin_type(plugin);
    const int32_t need = !type ? 0 : (std::strncmp(type, "SPConvIdx", 9) == 0 ? 3 : (std::strcmp(type, "SPConvMM") == 0 ? 5 : 4));
    if (nb_in < need) {
      d3d::setError("schedule: %s reads %d inputs, step names %d", type ? type : "?", need, nb_in);
      return D3D_ERR_BAD_ARG;
    }
  }
  if (nb_out != d3d_num_outputs(plugin)) {
    d3d::setError("schedule: %s has %d outputs, step names %d", d3d_plugin_type(plugin), d3d_num_outputs(plugin), nb_out);
    return D3D_ERR_BAD_ARG;
  }
  d3d_schedule::Step st;
  st.plugin = plugin;
  st.in.assign(in_desc, in_desc + nb_in);
  st.out.assign(out_desc, out_desc + nb_out);
  st.inputs.assign(inputs, inputs + nb_in);
  st.outputs.assign(outputs, outputs + nb_out);
  st.workspace = workspace;
  st.workspaceBytes = workspace_bytes;
  st.lane = lane;
  return appendStep(s, std::move(st), after, nb_after);
  D3D_GUARD_END(D3D_ERR_BAD_ARG)
}

int32_t d3d_schedule_add_sum(d3d_schedule* s, int32_t dtype, const void* a, const void* b, void* out, int64_t count,
                             int32_t lane, const int32_t* after, int32_t nb_after) {
  D3D_GUARD_BEGIN
  if (!s || count < 0 || (count && (!a || !b || !out))) {
    d3d::setError("schedule: bad sum (null tensor or negative count)");
    return D3D_ERR_BAD_ARG;
  }
  if (dtype != D3D_FLOAT && dtype != D3D_HALF && dtype != D3D_BF16) {
    d3d::setError("schedule: sums of dtype %d not implemented", dtype);
    return D3D_ERR_UNSUPPORTED;
  }
  d3d_schedule::Step st;
  st.kind = d3d_schedule::kSum;
  st.dtype = dtype;
  st.count = count;
  st.inputs = {a, b};
  st.outputs = {out};
  st.lane = lane;
  return appendStep(s, std::move(st), after, nb_after);
  D3D_GUARD_END(D3D_ERR_BAD_ARG)
}

int32_t d3d_schedule_add_cast(d3d_schedule* s, int32_t dtype, const void* a, void* out, int64_t count, int32_t lane,
                              const int32_t* after, int32_t nb_after) {
  D3D_GUARD_BEGIN
  if (!s || count < 0 || (count && (!a || !out))) {
    d3d::setError("schedule: bad cast (null tensor or negative count)");
    return D3D_ERR_BAD_ARG;
  }
  if (dtype != D3D_HALF && dtype != D3D_BF16) {
    d3d::setError("schedule: casts from float to dtype %d not implemented", dtype);
    return D3D_ERR_UNSUPPORTED;
  }
  d3d_schedule::Step st;
  st.kind = d3d_schedule::kCast;
  st.dtype = dtype;
  st.count = count;
  st.inputs = {a};
  st.outputs = {out};
  st.lane = lane;
  return appendStep(s, std::move(st), after, nb_after);
  D3D_GUARD_END(D3D_ERR_BAD_ARG)
}

int32_t d3d_schedule_run(d3d_schedule* s, void* stream) {
  D3D_GUARD_BEGIN
  if (!s) return D3D_ERR_BAD_ARG;
  hipStream_t main = static_cast<hipStream_t>(stream);
  // A run puts event edges between streams that are not the caller's; under stream capture that is a topology
  // this runtime has crashed on at the end of the capture.  d3d_schedule_capture captures the steps without any.
  hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(main, &cap) == hipSuccess && cap != hipStreamCaptureStatusNone) {
    d3d::setError("schedule: the stream is capturing; a schedule runs eagerly");
    return D3D_ERR_UNSUPPORTED;
  }
  reapGraphs(false);
  const uint64_t changes = changesOf(s);
  s->steady = s->lastChanges == changes ? s->steady + 1 : 0;
  if (s->steady >= s->patience && !(s->graph && s->graphChanges == changes)) {
    // what the operators enqueue is settled, and the pass repeats: capturing it costs about what one pass does
    dropGraph(s, main);
    const bool captured = captureGraph(s);
    s->graphChanges = changes;
    if (captured && changesOf(s) == changes) {
      s->patience = d3d_schedule::kSteadyRuns;
    } else {  // refused, which may pass (memory, a capture in another thread), or an operator is not settled after all
      dropGraph(s, main);
      s->steady = 0;
      s->patience = std::min(2 * s->patience, d3d_schedule::kMostPatience);
    }
  }
  if (s->graph && s->graphChanges == changes) {
    s->lastChanges = changes;
    const hipError_t launched = hipGraphLaunch(s->graph, main);
    if (launched != hipSuccess) return hipFail(launched, "hipGraphLaunch");
    s->launched = true;
    s->launchedOn = main;  // runs use the same tensors, so the caller orders them: the last launch is the last to end
    return D3D_OK;
  }
  hipError_t e = makeLanes(s);
  if (e != hipSuccess) return hipFail(e, "creating streams and events");
  auto laneStream = [&](int lane) { return lane == 0 ? main : s->lanes[static_cast<size_t>(lane)]; };
  if (s->lanes.size() > 1) {
    e = hipEventRecord(s->fork, main);
    for (size_t l = 1; l < s->lanes.size() && e == hipSuccess; ++l) e = hipStreamWaitEvent(s->lanes[l], s->fork, 0);
    if (e != hipSuccess) return hipFail(e, "fork");
  }
  int32_t rc = D3D_OK;
  for (auto& st : s->steps) {
    hipStream_t q = laneStream(st.lane);
    for (int dep : st.after) {
      e = hipStreamWaitEvent(q, s->steps[static_cast<size_t>(dep)].done, 0);
      if (e != hipSuccess && rc == D3D_OK) rc = hipFail(e, "hipStreamWaitEvent");
    }
    if (rc == D3D_OK)  // after a failure nothing more is enqueued, but the lanes still join below
      rc = d3d::scheduleEnqueueStep(st, q);
    if (st.done) {
      e = hipEventRecord(st.done, q);
      if (e != hipSuccess && rc == D3D_OK) rc = hipFail(e, "hipEventRecord");
    }
  }
  for (size_t l = 1; l < s->lanes.size(); ++l) {
    e = hipEventRecord(s->joined[l], s->lanes[l]);
    if (e == hipSuccess) e = hipStreamWaitEvent(main, s->joined[l], 0);
    if (e != hipSuccess && rc == D3D_OK) rc = hipFail(e, "join");
  }
  const uint64_t now = changesOf(s);
  if (rc != D3D_OK || now != changes) s->steady = 0;
  s->lastChanges = rc == D3D_OK ? now : ~0ull;
  return rc;
  D3D_GUARD_END(D3D_ERR_BAD_ARG)
}

int32_t d3d_schedule_size(const d3d_schedule* s) { return s ? static_cast<int32_t>(s->steps.size()) : D3D_ERR_BAD_ARG; }

}  // extern "C"
