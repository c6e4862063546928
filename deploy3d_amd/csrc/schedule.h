// A recorded pass (schedule.cpp) and what its two ways into a graph share.
#pragma once
#include <hip/hip_runtime.h>

#include <vector>

#include "common.h"
#include "d3d_spconv.h"

struct d3d_schedule {
  enum Kind { kOperator, kSum, kCast };
  struct Step {
    Kind kind = kOperator;
    d3d_plugin* plugin = nullptr;
    int32_t dtype = 0;          // kSum, kCast
    int64_t count = 0;
    std::vector<d3d_tensor_desc> in, out;
    std::vector<const void*> inputs;
    std::vector<void*> outputs;
    void* workspace = nullptr;
    size_t workspaceBytes = 0;
    int lane = 0;
    std::vector<int> after;     // steps of other lanes it waits for
    int before = -1;            // the step ahead of it on its own lane
    bool awaited = false;       // a step of another lane waits for it ...
    hipEvent_t done = nullptr;  // ... through this, recorded behind it
  };
  // made by the first run that enqueues step by step: a schedule that is only captured needs no stream and no event
  std::vector<hipStream_t> lanes;  // [0] unused: lane 0 is the caller's stream
  std::vector<hipEvent_t> joined;  // per owned lane: its tail, for the join
  hipEvent_t fork = nullptr;
  std::vector<Step> steps;
  // the pass as a graph
  hipGraphExec_t graph = nullptr;
  bool launched = false;        // the graph has been launched, last on launchedOn
  hipStream_t launchedOn = nullptr;
  uint64_t graphChanges = 0;    // the operators' change count the graph was captured at
  uint64_t lastChanges = ~0ull; // ... and at the end of the last run
  int steady = 0;               // runs in a row that changed nothing
  int patience = kSteadyRuns;   // ... after which a capture is tried; doubled by every refusal, as it costs a pass
  static constexpr int kSteadyRuns = 2, kMostPatience = 4096;
};

namespace d3d {

int32_t scheduleEnqueueStep(const d3d_schedule::Step& st, hipStream_t q);
// Per step the steps it directly comes behind (its lane's previous one and those it names), without those that are implied.
std::vector<std::vector<int>> scheduleEdges(const d3d_schedule* s);

}  // namespace d3d
