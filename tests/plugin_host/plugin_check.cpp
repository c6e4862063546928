// Host check of csrc/plugin.cpp against a stand-in for the HIP runtime that remembers what was freed and stand-ins for the
// kernels that remember what they were handed: memory whose address a captured graph holds stays where it is.  No GPU.
#include <hip/hip_runtime.h>

#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <set>
#include <vector>

#include "common.h"
#include "d3d_spconv.h"

namespace {
std::set<void*> freed;
const int32_t* derivedTable = nullptr;   // the table of the last launchBuildNeighbours
d3d::ConvArgs lastConv;                  // of the last launchConv
bool capturing = false;
int sorts = 0;                           // launchOrderRows so far
int padTo = 0;                           // channels that narrow layers are widened to (0: they are not)
}  // namespace

// ---- the runtime: nothing is given back, so an address names one allocation ----
extern "C" {
const char* hipGetErrorString(hipError_t) { return "stand-in error"; }
hipError_t hipMalloc(void** p, size_t n) {
  *p = std::aligned_alloc(256, (n + 255) / 256 * 256);
  return *p ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipFree(void* p) {
  freed.insert(p);
  return hipSuccess;
}
hipError_t hipMemcpy(void* to, const void* from, size_t n, hipMemcpyKind) {
  std::memcpy(to, from, n);
  return hipSuccess;
}
hipError_t hipMemset(void* p, int v, size_t n) {
  std::memset(p, v, n);
  return hipSuccess;
}
hipError_t hipGetDevice(int* d) {
  *d = 0;
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus* st) {
  *st = capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
  return hipSuccess;
}
}
// ---- the kernels ----
namespace d3d {
int32_t launchConv(const ConvArgs& a, hipStream_t) {
  lastConv = a;
  return D3D_OK;
}
int32_t launchBuildNeighbours(const int32_t*, int64_t, const int32_t*, bool, int, int64_t, int64_t, int32_t* nbr, hipStream_t) {
  derivedTable = nbr;
  return D3D_OK;
}
int32_t launchOrderRows(int32_t*, int, int64_t, const int32_t*, const RowOrder&, hipStream_t) {
  ++sorts;
  return D3D_OK;
}
size_t orderRowsBytes(int64_t outRows) { return static_cast<size_t>(outRows) * 5 + 128; }
RowOrder orderRowsAt(void* base, int64_t) { return {static_cast<int32_t*>(base), static_cast<unsigned long long*>(base)}; }
bool convTakesRowOrder(const ConvArgs&) { return true; }
bool convUsesMfma(int32_t, int cin, int cout) { return cin % 16 == 0 && cout % 16 == 0; }
bool floatMfmaFits(int, int, int) { return true; }
int paddedMfmaChannels(int32_t, int cin, int) { return padTo > cin ? padTo : cin; }
bool convReadsNarrowRows(int32_t, int, int, int, int64_t) { return false; }
int32_t launchPadRows(const void*, int64_t, int, int, void*, hipStream_t) { return D3D_OK; }
int32_t launchRulebook(const RbGeom&, bool, const int32_t*, const int32_t*, int64_t, int32_t, int32_t*, int32_t*, int32_t*, int32_t*,
                       void*, size_t, RbSide&, hipStream_t) {
  return D3D_OK;
}
size_t rulebookWorkspaceBytes(const RbGeom&, int64_t, bool, bool) { return 256; }
size_t mapStateWords(size_t) { return 64; }
void blockMapBytes(const RbGeom&, int64_t, size_t* records, size_t* chunkBase) { *records = *chunkBase = 0; }
int32_t launchDensify(const DensifyArgs&, hipStream_t) { return D3D_OK; }
size_t densifyWorkspaceBytes(int64_t, int64_t, int64_t, int64_t) { return 256; }
int32_t launchVoxelize(const VoxelizeArgs&, hipStream_t) { return D3D_OK; }
size_t voxelizeWorkspaceBytes(int64_t, int64_t, int64_t) { return 256; }
int32_t staticScratch(void**, size_t*) { return D3D_ERR_UNSUPPORTED; }
}  // namespace d3d

#define CHECK(cond)                                                               \
  do {                                                                            \
    if (!(cond)) {                                                                \
      std::fprintf(stderr, "plugin_check: %s failed (line %d)\n", #cond, __LINE__); \
      return 1;                                                                   \
    }                                                                             \
  } while (0)

namespace {
constexpr int32_t kTypes[4] = {D3D_HALF, D3D_INT8, D3D_BF16, D3D_FLOAT};

struct Conv {
  d3d_plugin* plugin = nullptr;
  int32_t cin, cout, rows;
  d3d_tensor_desc in[5], out[1];
  alignas(256) unsigned char memory[256];
  Conv(int32_t kVol, int32_t cin_, int32_t cout_, int32_t rows_, bool inverse) : cin(cin_), cout(cout_), rows(rows_) {
    std::vector<unsigned char> blob(19 + static_cast<size_t>(kVol) * cin * cout * 4, 0);
    const int32_t head[4] = {kVol, cin, cout, rows};
    std::memcpy(blob.data(), head, 16);
    blob[16] = inverse ? 0 : 1;
    blob[17] = inverse ? 1 : 0;
    d3d_create("SPConvMM", "2.0", blob.data(), blob.size(), &plugin);
    std::memset(in, 0, sizeof(in));
    std::memset(out, 0, sizeof(out));
    auto shape = [](d3d_tensor_desc* d, int32_t dtype, int32_t nb, int64_t a, int64_t b) {
      d->dtype = dtype;
      d->nb_dims = nb;
      d->dims[0] = a;
      d->dims[1] = b;
    };
    shape(&in[0], D3D_HALF, 2, rows, cin);
    shape(&in[1], D3D_INT32, 1, 1, 0);
    shape(&in[2], D3D_INT32, 1, 1, 0);
    shape(&in[3], D3D_INT32, 2, 3, static_cast<int64_t>(kVol) * (rows + 128));
    shape(&in[4], D3D_INT32, 1, 1, 0);
    shape(&out[0], D3D_HALF, 2, rows, cout);
  }
  ~Conv() { d3d_destroy(plugin); }
  void type(int32_t dtype) { in[0].dtype = out[0].dtype = dtype; }
  int32_t configure() { return d3d_configure(plugin, in, 5, out, 1); }
  int32_t enqueue() {
    const void* ins[5] = {memory, memory, memory, memory, memory};
    void* outs[1] = {memory};
    return d3d_enqueue(plugin, in, out, ins, outs, nullptr, 0, nullptr);
  }
};

// The table a layer derives is at one address whatever feature types run: a captured enqueue of one type writes and reads it on
// every replay.
int derivedTableStays() {
  for (int32_t first : kTypes)
    for (int inverse = 0; inverse < 2; ++inverse)
      for (int32_t kVol : {1, 8, 27, 32, 45})
        for (int configured = 0; configured < 2; ++configured) {
          Conv c(kVol, 64, 64, 2000, inverse != 0);
          CHECK(c.plugin);
          c.type(first);
          if (configured) CHECK(c.configure() == D3D_OK);
          CHECK(c.enqueue() == D3D_OK);
          capturing = true;
          CHECK(c.enqueue() == D3D_OK);
          capturing = false;
          const int32_t* const table = derivedTable;
          for (int32_t t : kTypes) {
            c.type(t);
            if (configured) CHECK(c.configure() == D3D_OK);
            CHECK(c.enqueue() == D3D_OK);
            CHECK(derivedTable == table && !freed.count(const_cast<int32_t*>(table)));
          }
        }
  return 0;
}

// So are the rows of a narrow layer that one type widens, whatever the others need.
int widenedRowsStay() {
  for (int32_t first : kTypes)
    for (int configured = 0; configured < 2; ++configured) {
      padTo = 16;
      Conv c(27, 5, 16, 2000, false);
      CHECK(c.plugin);
      c.type(first);
      if (configured) CHECK(c.configure() == D3D_OK);
      CHECK(c.enqueue() == D3D_OK);
      const void* const rows = lastConv.in;
      CHECK(rows != c.memory && lastConv.cin == 16);
      for (int32_t t : kTypes) {
        c.type(t);
        if (configured) CHECK(c.configure() == D3D_OK);
        CHECK(c.enqueue() == D3D_OK);
        CHECK(lastConv.in == rows && !freed.count(const_cast<void*>(rows)));
      }
      padTo = 0;
    }
  return 0;
}

// Which layers sort the rows of their derived table: those that were measured to gain by it, on both sides of each line.
int sortedLayers() {
  struct Layer {
    int32_t dtype, kVol, cin, cout, rows;
    bool inverse, sorted;
  };
  const Layer layers[] = {
      {D3D_FLOAT, 27, 64, 32, 300, true, true},      {D3D_FLOAT, 27, 32, 16, 2000, true, false},   {D3D_FLOAT, 27, 32, 16, 2100, true, true},
      {D3D_FLOAT, 27, 32, 32, 30000, true, false},   {D3D_FLOAT, 27, 32, 32, 40000, true, true},   {D3D_FLOAT, 27, 16, 16, 60000, true, false},
      {D3D_FLOAT, 27, 16, 32, 4000, true, true},     {D3D_FLOAT, 27, 16, 128, 60000, true, false}, {D3D_FLOAT, 4, 64, 32, 9000, true, false},
      {D3D_FLOAT, 36, 64, 32, 9000, true, false},    {D3D_FLOAT, 27, 32, 32, 8000, false, true},   {D3D_FLOAT, 27, 32, 32, 30000, false, false},
      {D3D_FLOAT, 27, 32, 32, 110000, false, true},  {D3D_FLOAT, 27, 64, 32, 16000, false, true},  {D3D_FLOAT, 27, 64, 32, 60000, false, false},
      {D3D_FLOAT, 27, 64, 64, 30000, false, true},   {D3D_FLOAT, 27, 16, 32, 4000, false, false},  {D3D_HALF, 27, 32, 16, 300, true, true},
      {D3D_HALF, 27, 64, 32, 100000, true, false},   {D3D_BF16, 27, 64, 64, 100000, true, false},  {D3D_BF16, 27, 128, 128, 60000, true, false},
      {D3D_BF16, 27, 128, 128, 75000, true, true},   {D3D_HALF, 27, 64, 128, 110000, true, false}, {D3D_HALF, 27, 64, 128, 140000, true, true},
      {D3D_HALF, 27, 128, 128, 110000, false, false}, {D3D_INT8, 27, 64, 64, 30000, true, false},  {D3D_INT8, 27, 128, 128, 110000, true, false},
  };
  for (const Layer& l : layers) {
    Conv c(l.kVol, l.cin, l.cout, l.rows, l.inverse);
    CHECK(c.plugin);
    c.type(l.dtype);
    sorts = 0;
    CHECK(c.enqueue() == D3D_OK);
    if (sorts != (l.sorted ? 1 : 0)) std::fprintf(stderr, "dtype %d, %d -> %d, %d rows, inverse %d\n", l.dtype, l.cin, l.cout, l.rows, l.inverse);
    CHECK(sorts == (l.sorted ? 1 : 0) && (lastConv.rowOrder != nullptr) == l.sorted);
  }
  return 0;
}
}  // namespace

int main() {
  if (derivedTableStays() || widenedRowsStay() || sortedLayers()) return 1;
  std::puts("plugin_check ok");
  return 0;
}
