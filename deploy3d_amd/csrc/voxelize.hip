// Points -> voxels with mean features (the step in front of a sparse backbone).
//
// Reference: voxel_encoder::func::simpleMeanEncoder and its kernels,
// trt/voxel_encoder/simple_mean_trt.cu:26-168.  A point is kept when all its
// features are finite, its batch index is not negative and its cell
//   (b, int((z - zMin) / zSize), int((y - yMin) / ySize), int((x - xMin) / xSize))
// (fp32 arithmetic, conversion truncating toward zero) lies in the grid; every
// occupied cell becomes one output row holding the mean of its points' features,
// its coordinate, and numActOut = min(occupied cells, maxNumActOut).
//
// The reference numbers the voxels in hash-slot order, which depends on the
// races of its insertions.  Here a voxel is represented by the lowest index
// among its points (a 64-bit atomic min on key<<32 | index, so the table's
// races cannot show), and voxels are numbered by a prefix sum over the points
// of "I am my voxel's representative": rows come out in order of first
// appearance, the same on every run, and truncation keeps the voxels that
// appear first.  Sums use fp32 atomic adds like the reference's, so the means
// can differ in the last bits from run to run; coordinates and counts cannot.
//
// Three forms, chosen by size (launchVoxelize): a few thousand points fit one workgroup's LDS (one launch); otherwise
// records of the points carry the sums (three launches: clear, insert, emit); very many points or channels keep a table
// of bare keys and sum in the output rows (five launches).
#include <atomic>

#include "common.h"

namespace d3d {
namespace {

constexpr int kVxThreads = 256;
constexpr int kVxItems = 4;
constexpr int kVxChunk = kVxThreads * kVxItems;  // points per workgroup of the ranking pass
constexpr uint32_t kVxNone = 0xFFFFFFFFu;
constexpr unsigned long long kVxEmpty = ~0ull;

// trt/include/common/hash32.h:23-33 (MurmurHash3 finaliser)
__device__ __forceinline__ uint32_t vxMix(uint32_t k) {
  k ^= k >> 16;
  k *= 0x85ebca6bu;
  k ^= k >> 13;
  k *= 0xc2b2ae35u;
  k ^= k >> 16;
  return k;
}

struct VxGeom {
  int B, Z, Y, X;
};

// Features of a point: CT channels in registers (0 = any number, left in memory).  All loads are requested before the
// first value is looked at - a chain of loads that each wait for the check of the one before cost a small call 10 us.
template <int CT> struct VxPoint {
  float v[CT ? CT : 3];
  const float* p;
  bool finite;
  __device__ __forceinline__ VxPoint(const float* f, int C) : p(f) {
    uint32_t worst = 0;   // largest exponent field
#pragma unroll
    for (int c = 0; c < (CT ? CT : 3); ++c) v[c] = f[c];
    if constexpr (CT == 0)
      for (int c = 3; c < C; ++c) worst = max(worst, __float_as_uint(f[c]) & 0x7F800000u);
#pragma unroll
    for (int c = 0; c < (CT ? CT : 3); ++c) worst = max(worst, __float_as_uint(v[c]) & 0x7F800000u);
    finite = worst != 0x7F800000u;
  }
  __device__ __forceinline__ float operator[](int c) const { return CT ? v[c] : p[c]; }
};

// int((v - lo) / size) of IEEE division, usually without the division: the product with the reciprocal is off by a few
// units in the last place, which cannot change the integer part unless the product is that close to an integer.
__device__ __forceinline__ int vxAxis(float v, float lo, float size, float rcp) {
  const float d = v - lo, q = d * rcp;
  const float away = fabsf(q - rintf(q));
  // 2^-21 |q| is four times the error bound (2 ulp); small quotients, overflows and odd sizes take the division
  return (away > fabsf(q) * 4.76837158e-7f && fabsf(q) > 1e-3f && fabsf(q) < 1e6f && rcp < 1e30f && rcp > 1e-30f)
             ? static_cast<int>(q)
             : static_cast<int>(d / size);
}

struct VxConfig {
  float lo[3], size[3], rcp[3];
  __device__ __forceinline__ explicit VxConfig(const float* config) {
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      lo[q] = config[q];
      size[q] = config[3 + q];
      rcp[q] = 1.f / size[q];
    }
  }
};

// The cell of a point (simple_mean_trt.cu:36-52); false when a feature is not finite, the point is skipped or it lies
// outside the grid.
template <int CT>
__device__ __forceinline__ bool vxCell(const VxPoint<CT>& f, int b, const VxConfig& v, const VxGeom& g, uint32_t* key) {
  if (!f.finite || b < 0 || b >= g.B) return false;
  const int x = vxAxis(f.v[0], v.lo[0], v.size[0], v.rcp[0]);
  const int y = vxAxis(f.v[1], v.lo[1], v.size[1], v.rcp[1]);
  const int z = vxAxis(f.v[2], v.lo[2], v.size[2], v.rcp[2]);
  if (!(x >= 0 && x < g.X && y >= 0 && y < g.Y && z >= 0 && z < g.Z)) return false;
  *key = ((static_cast<uint32_t>(b) * g.Z + z) * g.Y + y) * g.X + x;
  return true;
}

// (b, z, y, x) of a cell (refnd.h:56-64)
__device__ __forceinline__ int4 vxCoord(uint32_t key, const VxGeom& g) {
  const uint32_t x = key % g.X;
  key /= g.X;
  const uint32_t y = key % g.Y;
  key /= g.Y;
  const uint32_t z = key % g.Z;
  return make_int4(static_cast<int>(key / g.Z), static_cast<int>(z), static_cast<int>(y), static_cast<int>(x));
}

// ---------------------------------------------------------------------------
// A few thousand points: table, sums and counts in the LDS of one workgroup.  Such a call is launch latency, on the
// host (3 us per launch) and on the device: at 3 001 points one launch of 10.8 us instead of five of 17.  Bound by one
// CU's instruction rate (16 wavefronts, about 22 000 cycles).  Workgroups past the first zero the output rows that no
// point can reach.  Up to 4096 points: 13 us a call there, 18 with the three launches below; four points per thread
// are also what the registers of 16 wavefronts hold.
// ---------------------------------------------------------------------------
constexpr int kVxSmallThreads = 1024;
constexpr int kVxSmallItems = 4;

template <int CT>
__global__ void __launch_bounds__(kVxSmallThreads)
vxSmall(const float* __restrict__ feats, const int32_t* __restrict__ batchIdx, const float* __restrict__ config, int32_t n,
        int channels, VxGeom g, uint32_t mask, int32_t maxNumActOut, float* __restrict__ outFeats, int32_t* __restrict__ outCoors,
        int32_t* __restrict__ numActOut) {
  extern __shared__ __attribute__((aligned(16))) unsigned char vxSmem[];
  const int C = CT ? CT : channels;
  const int tid = threadIdx.x;
  if (blockIdx.x > 0) {
    const int64_t total = static_cast<int64_t>(maxNumActOut) * C;
    for (int64_t e = static_cast<int64_t>(n) * C + static_cast<int64_t>(blockIdx.x - 1) * kVxSmallThreads + tid; e < total;
         e += static_cast<int64_t>(gridDim.x - 1) * kVxSmallThreads)
      outFeats[e] = 0.f;
    return;
  }
  unsigned long long* table = reinterpret_cast<unsigned long long*>(vxSmem);  // [mask + 1] key << 32 | lowest point, then id
  // [C, n]: a channel's sums of neighbouring voxels in neighbouring banks.  A voxel's representative stores its own
  // features and the other points add to them: LDS float atomics run at about 3 lanes per clock, and with every point
  // adding they were half of the kernel's time.
  float* sums = reinterpret_cast<float*>(table + mask + 1);
  uint32_t* counts = reinterpret_cast<uint32_t*>(sums + n * C);               // [n]
  __shared__ uint32_t waveReps[kVxSmallItems][kVxSmallThreads / 64];
  uint32_t key[kVxSmallItems], slot[kVxSmallItems];
  // point loads are on their way while the LDS is cleared
  float pts[kVxSmallItems][CT ? CT : 1];
  int batch[kVxSmallItems];
  if constexpr (CT != 0) {
#pragma unroll
    for (int k = 0; k < kVxSmallItems; ++k) {
      const int i = min(k * kVxSmallThreads + tid, n - 1);   // (no branch around a load: all of them in flight together)
      batch[k] = batchIdx[i];
#pragma unroll
      for (int c = 0; c < CT; ++c) pts[k][c] = feats[static_cast<size_t>(i) * CT + c];
    }
  }
  for (uint32_t e = tid; e < (mask + 1) / 2; e += kVxSmallThreads) reinterpret_cast<uint4*>(table)[e] = make_uint4(~0u, ~0u, ~0u, ~0u);
  const VxConfig cfg(config);
#pragma unroll
  for (int k = 0; k < kVxSmallItems; ++k) {
    const int i = k * kVxSmallThreads + tid;
    slot[k] = kVxNone;
    if constexpr (CT != 0) {
      const VxPoint<CT> point(pts[k], CT);
      if (vxCell(point, i < n ? batch[k] : -1, cfg, g, &key[k])) slot[k] = 0u;
    } else if (i < n) {
      const VxPoint<0> point(feats + static_cast<size_t>(i) * C, C);
      if (vxCell(point, batchIdx[i], cfg, g, &key[k])) slot[k] = 0u;
    }
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < kVxSmallItems; ++k) {
    if (slot[k] == kVxNone) continue;
    const unsigned long long mine = (static_cast<unsigned long long>(key[k]) << 32) | static_cast<uint32_t>(k * kVxSmallThreads + tid);
    uint32_t s = vxMix(key[k]) & mask;
    for (uint32_t tries = 0; tries <= mask; ++tries) {
      const unsigned long long old = atomicCAS(&table[s], kVxEmpty, mine);
      if (old == kVxEmpty) break;
      if (static_cast<uint32_t>(old >> 32) == key[k]) {
        if (old > mine) atomicMin(&table[s], mine);
        break;
      }
      s = (s + 1) & mask;
    }
    slot[k] = s;
  }
  __syncthreads();
  // voxel ids: representatives counted in point order
  const int lane = tid & 63, wave = tid >> 6;
  uint32_t below[kVxSmallItems];
  bool rep[kVxSmallItems];
#pragma unroll
  for (int k = 0; k < kVxSmallItems; ++k) {
    rep[k] = slot[k] != kVxNone && static_cast<uint32_t>(table[slot[k]]) == static_cast<uint32_t>(k * kVxSmallThreads + tid);
    const unsigned long long m = __ballot(rep[k]);
    below[k] = static_cast<uint32_t>(__popcll(m & ((1ull << lane) - 1ull)));
    if (lane == 0) waveReps[k][wave] = static_cast<uint32_t>(__popcll(m));
  }
  __syncthreads();
  uint32_t total = 0;
#pragma unroll
  for (int k = 0; k < kVxSmallItems; ++k) {
    uint32_t id = total + below[k];
#pragma unroll
    for (int w = 0; w < kVxSmallThreads / 64; ++w) {
      if (w < wave) id += waveReps[k][w];
      total += waveReps[k][w];
    }
    if (rep[k]) {
      reinterpret_cast<uint32_t*>(&table[slot[k]])[0] = id;
      if (id < static_cast<uint32_t>(maxNumActOut)) {
        reinterpret_cast<int4*>(outCoors)[id] = vxCoord(key[k], g);
        counts[id] = 1u;
        const float* f = feats + static_cast<size_t>(k * kVxSmallThreads + tid) * C;
        for (int c = 0; c < C; ++c) sums[c * n + id] = CT ? pts[k][c] : f[c];
      }
    }
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < kVxSmallItems; ++k) {
    if (slot[k] == kVxNone || rep[k]) continue;
    const uint32_t id = static_cast<uint32_t>(table[slot[k]]);
    if (id >= static_cast<uint32_t>(maxNumActOut)) continue;
    if constexpr (CT != 0) {
#pragma unroll
      for (int c = 0; c < CT; ++c) unsafeAtomicAdd(sums + c * n + id, pts[k][c]);
    } else {
      const float* f = feats + static_cast<size_t>(k * kVxSmallThreads + tid) * C;
      for (int c = 0; c < C; ++c) unsafeAtomicAdd(sums + c * n + id, f[c]);
    }
    atomicAdd(counts + id, 1u);
  }
  __syncthreads();
  const int rows = static_cast<int>(total < static_cast<uint32_t>(maxNumActOut) ? total : static_cast<uint32_t>(maxNumActOut));
  const int lastRow = n < maxNumActOut ? n : maxNumActOut;
  for (int r = tid; r < lastRow; r += kVxSmallThreads) {
    const bool live = r < rows;
    const float points = live ? static_cast<float>(counts[r]) : 1.f;
    if constexpr (CT == 4) {
      float mean[4];
#pragma unroll
      for (int c = 0; c < 4; ++c) mean[c] = live ? sums[c * n + r] / points : 0.f;
      __builtin_memcpy(outFeats + r * 4, mean, 16);
    } else {
      for (int c = 0; c < C; ++c) outFeats[r * C + c] = live ? sums[c * n + r] / points : 0.f;
    }
  }
  if (tid == 0) *numActOut = rows;
}

// ---------------------------------------------------------------------------
// The usual form: a table of heads, u64 key << 32 | the point that claimed the entry, and for every point a record that
// is its voxel's if it claimed one:
//   { u32 lowest point; float further points; float sums[C]; pad to 16 bytes }
// The lowest point's own features are not in the sums (most voxels of a scan hold one or two points, so most points
// then cost one compare-and-swap and no other atomic): the emitting pass reads them where they are.  A point that takes
// a higher one's place as the lowest adds the features of the point it displaced.  Records lie in point order: the
// emitting pass reads those of voxels with one point in one run, and heads of 8 bytes afford a table of four per point.
// (The count is exact: the form is for fewer than 2^24 points.)
// 200 000 points, 135 000 of them in the grid and nearly all in voxels of their own: clear 5.8, insert 11.8, emit 6.2 us, where
// entries of 32 bytes in a table of two per point took 8, 16.6 and 10.3: bound by the chains of compare-and-swaps, whose longest
// went from 16 to 9 with the larger table (eight heads per point: insert 10.0, but with eight points to a voxel the call is 1 us
// slower).  In a graph of calls 36.0 -> 22.8 us, 100 000 points 27.9 -> 16.9; eight points to a voxel 62 -> 28.8, 400 000 of them
// with six channels 136 -> 55.  Up to 50 000 points the call is bound by its three launches on the host.
// ---------------------------------------------------------------------------
constexpr int kVxMaxWide = 12;  // channels a record carries
constexpr int64_t kVxSmallChunks = 128 * 1024;  // most points of a call in chunks of 256 (see vxEmitWide)

__host__ __device__ constexpr int vxRecordBytes(int C) { return (8 + 4 * C + 15) / 16 * 16; }

// Heads empty, every record's lowest point its own, output rows zero (simple_mean_trt.cu:139-143), chunk states zero.
template <int PER>
__global__ void __launch_bounds__(kVxThreads)
vxClearWide(uint4* table, uint32_t headPairs, uint4* records, uint32_t pieces, float* outFeats, int64_t nFeats,
            unsigned long long* states, uint32_t nStates) {
  const int64_t stride = static_cast<int64_t>(gridDim.x) * blockDim.x;
  const int64_t tid = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  for (int64_t i = tid; i < headPairs; i += stride) table[i] = make_uint4(~0u, ~0u, ~0u, ~0u);
  for (uint32_t i = static_cast<uint32_t>(tid); i < pieces; i += static_cast<uint32_t>(stride))
    records[i] = make_uint4(i % PER == 0 ? i / PER : 0u, 0u, 0u, 0u);
  for (int64_t i = tid; i < nFeats; i += stride) outFeats[i] = 0.f;
  for (int64_t i = tid; i < nStates; i += stride) states[i] = 0ull;
}

// points[i] = { record of point i's voxel when i may be its lowest point, else none; key }.
template <int CT>
__global__ void __launch_bounds__(kVxThreads)
vxInsertWide(const float* __restrict__ feats, const int32_t* __restrict__ batchIdx, const float* __restrict__ config, int32_t n,
             int channels, VxGeom g, unsigned long long* table, uint32_t slots, unsigned char* records,
             uint2* __restrict__ points) {
  const int C = CT ? CT : channels;
  constexpr int W = CT ? 8 : 16;     // lanes that add a point: one for the count and one per channel
  static_assert(CT + 1 <= 8 && kVxMaxWide + 1 <= 16, "a lane per word");
  __shared__ float words[kVxThreads * W];
  __shared__ uint32_t homes[kVxThreads];
  const int32_t i = blockIdx.x * kVxThreads + threadIdx.x, at = min(i, n - 1);
  const VxPoint<CT> f(feats + static_cast<size_t>(at) * C, C);
  const VxConfig cfg(config);
  uint32_t key = 0, home = kVxNone, added = kVxNone;   // the voxel's record, and the point whose features go to its sums
  bool lowest = false;
  if (vxCell(f, i < n ? batchIdx[at] : -1, cfg, g, &key)) {
    const unsigned long long mine = (static_cast<unsigned long long>(key) << 32) | static_cast<uint32_t>(i);
    // the hash spread over the table by its high bits: any number of slots will do
    uint32_t s = static_cast<uint32_t>((static_cast<unsigned long long>(vxMix(key)) * slots) >> 32);
    for (uint32_t tries = 0; tries < slots; ++tries) {
      const unsigned long long old = atomicCAS(table + s, kVxEmpty, mine);
      if (old == kVxEmpty) {
        home = static_cast<uint32_t>(i);
        lowest = true;
        break;
      }
      if (static_cast<uint32_t>(old >> 32) == key) {
        home = static_cast<uint32_t>(old);
        added = static_cast<uint32_t>(i);
        if (added < home) {
          const uint32_t low = atomicMin(reinterpret_cast<uint32_t*>(records + static_cast<size_t>(home) * vxRecordBytes(C)), added);
          lowest = low > added;
          added = max(low, added);
        }
        break;
      }
      s = s + 1 == slots ? 0u : s + 1;
    }
  }
  if (i < n) points[i] = make_uint2(lowest ? home : kVxNone, key);
  // The words that a point adds are one run of 4 * (C + 1) bytes: neighbouring lanes add them together, a wavefront
  // instruction for 64 / W points, so that memory sees one access per point and not one per word.
  const unsigned long long adds = __ballot(added != kVxNone);
  const int lane = threadIdx.x & 63, first = threadIdx.x & ~63, count = __popcll(adds);
  if (added != kVxNone) {
    const int to = first + __popcll(adds & ((1ull << lane) - 1ull));
    homes[to] = home;
    words[to * W] = 1.f;
    const float* from = feats + static_cast<size_t>(added) * C;
    for (int c = 0; c < C; ++c) words[to * W + 1 + c] = from[c];
  }
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");   // a wavefront reads what it wrote itself
  __builtin_amdgcn_wave_barrier();
  const int w = lane % W;
  for (int p = lane / W; p < count; p += 64 / W)
    if (w <= C)
      unsafeAtomicAdd(reinterpret_cast<float*>(records + static_cast<size_t>(homes[first + p]) * vxRecordBytes(C) + 4) + w,
                      words[(first + p) * W + w]);
}

constexpr unsigned long long kVxPublished = 1ull << 32;
constexpr int kVxSpins = 1 << 16;

// One chunk of points per workgroup: representatives are ranked in point order, the workgroup publishes its count,
// reads how many the chunks before it have (a thread per chunk, so that all states are on their way together, waiting for
// those that are not there yet) and writes mean and coordinate of its own voxels.  A state is one 64-bit word, flag and
// value together, so relaxed device-scope accesses are enough.  The wait cannot deadlock - a chunk waits for lower ones
// only, and those were dispatched before it and wait for nobody before they publish - and it is bounded all the same:
// after kVxSpins looks the thread counts that chunk's representatives itself.
// The pass is a chain of loads (points, records, features, states), so small calls take chunks of 256 points, which fill the
// chip: in a graph of calls 10 000 points 13.8 us with chunks of 1024, 11.9 with 512, 10.9 with 256; 50 000 15.5, 13.8, 12.7;
// 100 000 18.2, 17.0, 16.9.  Every chunk reads the states of all before it: 200 000 points 23.8, 22.7, 23.1, 930 000 63.9, 63.4, 64.3
// (eight points to a voxel 93.8, 93.5, 96.7).  Hence 256 up to kVxSmallChunks points and 512 beyond.
template <int CT, int ITEMS>
__global__ void __launch_bounds__(kVxThreads)
vxEmitWide(const float* __restrict__ feats, int32_t n, int channels, VxGeom g, const unsigned char* __restrict__ records,
           const uint2* __restrict__ points, unsigned long long* states, int32_t maxNumActOut, float* __restrict__ outFeats,
           int32_t* __restrict__ outCoors, int32_t* __restrict__ numActOut) {
  constexpr int kChunk = kVxThreads * ITEMS;
  const int C = CT ? CT : channels;
  const size_t recordBytes = vxRecordBytes(C);
  __shared__ uint32_t waveReps[ITEMS][kVxThreads / 64], waveBase[kVxThreads / 64];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const uint32_t chunk = blockIdx.x;
  uint2 point[ITEMS];
  uint4 head[ITEMS];
  bool rep[ITEMS];
  uint32_t below[ITEMS];
#pragma unroll
  for (int k = 0; k < ITEMS; ++k) {
    const int64_t i = static_cast<int64_t>(chunk) * kChunk + k * kVxThreads + tid;
    point[k] = i < n ? points[i] : make_uint2(kVxNone, 0u);
  }
#pragma unroll
  for (int k = 0; k < ITEMS; ++k)
    head[k] = point[k].x != kVxNone ? *reinterpret_cast<const uint4*>(records + point[k].x * recordBytes) : make_uint4(0, 0, 0, 0);
#pragma unroll
  for (int k = 0; k < ITEMS; ++k) {
    rep[k] = point[k].x != kVxNone && head[k].x == chunk * kChunk + k * kVxThreads + tid;
    const unsigned long long m = __ballot(rep[k]);
    below[k] = static_cast<uint32_t>(__popcll(m & ((1ull << lane) - 1ull)));
    if (lane == 0) waveReps[k][wave] = static_cast<uint32_t>(__popcll(m));
  }
  __syncthreads();
  uint32_t total = 0, rank[ITEMS];
#pragma unroll
  for (int k = 0; k < ITEMS; ++k) {
    rank[k] = total + below[k];
#pragma unroll
    for (int w = 0; w < kVxThreads / 64; ++w) {
      if (w < wave) rank[k] += waveReps[k][w];
      total += waveReps[k][w];
    }
  }
  if (tid == 0) __hip_atomic_store(&states[chunk], kVxPublished | total, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  float mean[ITEMS][CT ? CT : 1];   // loaded ahead of the wait for the chunks before
  if constexpr (CT != 0) {
#pragma unroll
    for (int k = 0; k < ITEMS; ++k) {
      if (!rep[k]) continue;
      const float* f = feats + static_cast<size_t>(head[k].x) * CT;
      const float* sums = reinterpret_cast<const float*>(records + point[k].x * recordBytes + 8);
#pragma unroll
      for (int c = 0; c < CT; ++c) mean[k][c] = f[c] + (c == 0 ? __uint_as_float(head[k].z) : c == 1 ? __uint_as_float(head[k].w) : sums[c]);
    }
  }
  uint32_t base = 0;
  for (uint32_t p = tid; p < chunk; p += kVxThreads) {
    unsigned long long st = 0;
    for (int spins = 0; spins < kVxSpins; ++spins) {
      st = __hip_atomic_load(&states[p], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (st) break;
      __builtin_amdgcn_s_sleep(1);
    }
    if (!st)
      for (int64_t q = static_cast<int64_t>(p) * kChunk; q < static_cast<int64_t>(p + 1) * kChunk; ++q) {
        const uint32_t at = points[q].x;
        if (at != kVxNone && *reinterpret_cast<const uint32_t*>(records + at * recordBytes) == static_cast<uint32_t>(q)) ++st;
      }
    base += static_cast<uint32_t>(st);
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) base += __shfl_xor(base, off, 64);
  if (lane == 0) waveBase[wave] = base;
  __syncthreads();
  base = 0;
#pragma unroll
  for (int w = 0; w < kVxThreads / 64; ++w) base += waveBase[w];
  if (tid == 0 && chunk == gridDim.x - 1) *numActOut = static_cast<int32_t>(min(base + total, static_cast<uint32_t>(maxNumActOut)));
#pragma unroll
  for (int k = 0; k < ITEMS; ++k) {
    const uint32_t id = base + rank[k];
    if (!rep[k] || id >= static_cast<uint32_t>(maxNumActOut)) continue;
    float* row = outFeats + static_cast<size_t>(id) * C;
    const float count = __uint_as_float(head[k].y) + 1.f;
    if constexpr (CT != 0) {
#pragma unroll
      for (int c = 0; c < CT; ++c) row[c] = mean[k][c] / count;
    } else {
      const float* sums = reinterpret_cast<const float*>(records + point[k].x * recordBytes + 8);
      const float* f = feats + static_cast<size_t>(head[k].x) * C;
      for (int c = 0; c < C; ++c) row[c] = (f[c] + sums[c]) / count;
    }
    reinterpret_cast<int4*>(outCoors)[id] = vxCoord(point[k].y, g);
  }
}

// ---------------------------------------------------------------------------
// Very many points or channels: a table of keys, sums in the output rows.
// ---------------------------------------------------------------------------
// table = empty, outFeats = 0 (simple_mean_trt.cu:139-143), counts = 0, ticket = 0
__global__ void __launch_bounds__(kVxThreads)
vxReset(unsigned long long* table, int64_t slots, float* outFeats, int64_t nFeats, uint32_t* counts, int64_t nCounts,
        int32_t* numActOut) {
  const int64_t stride = static_cast<int64_t>(gridDim.x) * blockDim.x;
  const int64_t tid = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  for (int64_t i = tid; i < slots; i += stride) table[i] = kVxEmpty;
  for (int64_t i = tid; i < nFeats; i += stride) outFeats[i] = 0.f;
  for (int64_t i = tid; i < nCounts; i += stride) counts[i] = 0;
  if (tid == 0) *numActOut = 0;
}

// kernel::voxelize (simple_mean_trt.cu:28-60).  pointSlot[i] = the slot of point i's voxel, or none.
__global__ void __launch_bounds__(kVxThreads)
vxInsert(const float* __restrict__ feats, const int32_t* __restrict__ batchIdx, const float* __restrict__ config, int32_t n,
         int C, VxGeom g, unsigned long long* table, uint32_t mask, uint32_t* __restrict__ pointSlot) {
  const int32_t i = blockIdx.x * kVxThreads + threadIdx.x;
  if (i >= n) return;
  const VxConfig cfg(config);
  uint32_t key, slot = kVxNone;
  if (vxCell(VxPoint<0>(feats + static_cast<size_t>(i) * C, C), batchIdx[i], cfg, g, &key)) {
    const unsigned long long mine = (static_cast<unsigned long long>(key) << 32) | static_cast<uint32_t>(i);
    uint32_t s = vxMix(key) & mask;
    for (uint32_t tries = 0; tries <= mask; ++tries) {  // at most half the slots are ever taken
      const unsigned long long old = atomicCAS(&table[s], kVxEmpty, mine);
      if (old == kVxEmpty) {
        slot = s;
        break;
      }
      if (static_cast<uint32_t>(old >> 32) == key) {
        if (old > mine) atomicMin(&table[s], mine);
        slot = s;
        break;
      }
      s = (s + 1) & mask;
    }
  }
  pointSlot[i] = slot;
}

// Numbers the voxels: a point that is the lowest of its voxel counts 1.  local[i] = how many such points
// precede i inside its chunk of 1024 points; chunk totals become exclusive chunk bases in the workgroup that
// finishes last (ticket counter, no waiting), which also writes numActOut (simple_mean_trt.cu:149-150, :87).
__global__ void __launch_bounds__(kVxThreads)
vxRank(const unsigned long long* __restrict__ table, const uint32_t* __restrict__ pointSlot, int32_t n,
       uint32_t* __restrict__ local, uint32_t* chunkBase, uint32_t nChunks, uint32_t* ticket, int32_t* numActOut,
       int32_t maxNumActOut) {
  __shared__ uint32_t scratch[kVxThreads / 64];
  __shared__ uint32_t isLast;
  const int32_t first = blockIdx.x * kVxChunk + threadIdx.x * kVxItems;
  uint32_t flag[kVxItems];
  uint32_t mine = 0;
#pragma unroll
  for (int j = 0; j < kVxItems; ++j) {
    const int32_t i = first + j;
    flag[j] = 0;
    if (i < n) {
      const uint32_t s = pointSlot[i];
      if (s != kVxNone && static_cast<uint32_t>(table[s]) == static_cast<uint32_t>(i)) flag[j] = 1;
    }
    mine += flag[j];
  }
  // exclusive prefix over the workgroup
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  uint32_t incl = mine;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const uint32_t up = __shfl_up(incl, off, 64);
    if (lane >= off) incl += up;
  }
  if (lane == 63) scratch[wave] = incl;
  __syncthreads();
  uint32_t rank = incl - mine, total = 0;
#pragma unroll
  for (int w = 0; w < kVxThreads / 64; ++w) {
    if (w < wave) rank += scratch[w];
    total += scratch[w];
  }
#pragma unroll
  for (int j = 0; j < kVxItems; ++j) {
    if (flag[j]) local[first + j] = rank;
    rank += flag[j];
  }
  if (threadIdx.x == 0) {
    // the total is published with a returning device-scope atomic (performed where every XCD sees it once the
    // result is back); only then is the ticket taken.  An acquire-release ticket instead (a device-scope release
    // per workgroup) measured 8.2 -> 13.8 us for this kernel on 100 000 points.
    uint32_t old = __hip_atomic_exchange(&chunkBase[blockIdx.x], total, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    asm volatile("s_waitcnt vmcnt(0)" : "+v"(old)::"memory");
    isLast = __hip_atomic_fetch_add(ticket, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == nChunks - 1 ? 1u : 0u;
  }
  __syncthreads();
  if (!isLast) return;
  uint32_t running = 0;
  for (uint32_t base = 0; base < nChunks; base += kVxThreads) {
    const uint32_t q = base + threadIdx.x;
    const uint32_t v = q < nChunks ? __hip_atomic_load(&chunkBase[q], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0u;
    uint32_t inc = v;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const uint32_t up = __shfl_up(inc, off, 64);
      if (lane >= off) inc += up;
    }
    __syncthreads();
    if (lane == 63) scratch[wave] = inc;
    __syncthreads();
    uint32_t before = running, sum = 0;
#pragma unroll
    for (int w = 0; w < kVxThreads / 64; ++w) {
      if (w < wave) before += scratch[w];
      sum += scratch[w];
    }
    if (q < nChunks) chunkBase[q] = before + inc - v;
    running += sum;
  }
  if (threadIdx.x == 0)
    *numActOut = static_cast<int32_t>(running < static_cast<uint32_t>(maxNumActOut) ? running : maxNumActOut);
}

// kernel::scatterAddFeats (simple_mean_trt.cu:62-91): sums, point counts, and the coordinate row, written by the
// voxel's representative (refnd.h:56-64 turns the cell offset back into (b, z, y, x)).
__global__ void __launch_bounds__(kVxThreads)
vxAccumulate(const float* __restrict__ feats, int32_t n, int C, VxGeom g, const unsigned long long* __restrict__ table,
             const uint32_t* __restrict__ pointSlot, const uint32_t* __restrict__ local,
             const uint32_t* __restrict__ chunkBase, int32_t maxNumActOut, float* outFeats, uint32_t* counts,
             int32_t* __restrict__ outCoors) {
  const int32_t i = blockIdx.x * kVxThreads + threadIdx.x;
  if (i >= n) return;
  const uint32_t s = pointSlot[i];
  if (s == kVxNone) return;
  const unsigned long long entry = table[s];
  const uint32_t rep = static_cast<uint32_t>(entry);
  const uint32_t id = chunkBase[rep / kVxChunk] + local[rep];
  if (id >= static_cast<uint32_t>(maxNumActOut)) return;
  const float* f = feats + static_cast<size_t>(i) * C;
  float* row = outFeats + static_cast<size_t>(id) * C;
  for (int c = 0; c < C; ++c) unsafeAtomicAdd(row + c, f[c]);
  atomicAdd(counts + id, 1u);
  if (rep == static_cast<uint32_t>(i))
    reinterpret_cast<int4*>(outCoors)[id] = vxCoord(static_cast<uint32_t>(entry >> 32), g);
}

// kernel::meanFeats (simple_mean_trt.cu:93-101)
__global__ void __launch_bounds__(kVxThreads)
vxMean(float* outFeats, const uint32_t* __restrict__ counts, const int32_t* __restrict__ numActOut, int C) {
  const int64_t total = static_cast<int64_t>(*numActOut) * C;
  const int64_t stride = static_cast<int64_t>(gridDim.x) * blockDim.x;
  for (int64_t q = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; q < total; q += stride)
    outFeats[q] = outFeats[q] / static_cast<float>(counts[q / C]);
}

uint32_t pow2AtLeast(uint64_t v) {
  uint32_t p = 1024;
  while (p < v && p < 0x80000000u) p <<= 1;
  return p;
}

size_t alignUp256(size_t v) { return (v + 255) & ~static_cast<size_t>(255); }

struct VxPlan {
  bool wide;              // records carry the sums
  uint32_t slots, nChunks;
  size_t table, records, pointSlot, local, chunkBase, counts, ticket, total;
};

// Records are cleared and heads are 8 bytes (72 bytes per point at 3 to 6 channels, 56 with two heads per point), so the form
// is kept to what the fixed scratch array of d3d_enqueue_static holds: about 1.2 million points at 3 to 6 channels.  Four heads per
// point: the longest chain of taken slots decides the inserting pass (see above).
VxPlan planVoxelize(int64_t numPts, int64_t maxNumActOut, int64_t C) {
  VxPlan p{};
  const int64_t n = numPts < 1 ? 1 : numPts;
  p.nChunks = static_cast<uint32_t>((n + kVxChunk - 1) / kVxChunk);
  if (C <= kVxMaxWide && n < (1 << 30)) {
    p.wide = true;
    for (int64_t perPoint = 4; perPoint >= 2; perPoint /= 2) {  // the reference's hashSpace = 2 (simple_mean_trt.cu:110)
      p.slots = static_cast<uint32_t>(perPoint * n < 1024 ? 1024 : perPoint * n);
      size_t off = alignUp256(static_cast<size_t>(p.slots) * 8);
      p.records = off;
      off = alignUp256(off + static_cast<size_t>(n) * vxRecordBytes(static_cast<int>(C)));
      const int64_t chunk = kVxThreads * (n <= kVxSmallChunks ? 1 : 2);
      p.nChunks = static_cast<uint32_t>((n + chunk - 1) / chunk);
      p.pointSlot = off;  // record and key of every point
      off = alignUp256(off + static_cast<size_t>(n) * 8);
      p.chunkBase = off;  // chunk states, u64
      off = alignUp256(off + static_cast<size_t>(p.nChunks) * 8);
      p.total = off;
      if (p.total <= kStaticScratchBytes) return p;
    }
    p = VxPlan{};
    p.nChunks = static_cast<uint32_t>((n + kVxChunk - 1) / kVxChunk);
  }
  p.slots = pow2AtLeast(static_cast<uint64_t>(n) * 2);
  size_t off = 0;
  p.table = off;
  off = alignUp256(off + static_cast<size_t>(p.slots) * 8);
  p.pointSlot = off;
  off = alignUp256(off + static_cast<size_t>(n) * 4);
  p.local = off;
  off = alignUp256(off + static_cast<size_t>(n) * 4);
  p.chunkBase = off;
  off = alignUp256(off + static_cast<size_t>(p.nChunks) * 4);
  p.counts = off;  // [maxNumActOut] point counts, directly followed by the ticket
  off += static_cast<size_t>(maxNumActOut < 0 ? 0 : maxNumActOut) * 4;
  p.ticket = off;
  off = alignUp256(off + 4);
  p.total = off;
  return p;
}

// One workgroup's form: at most kVxSmallItems points per thread, table and sums within a CU's LDS.
bool smallFits(int64_t numPts, int64_t C, uint32_t* slots, size_t* lds) {
  if (numPts < 1 || numPts > kVxSmallThreads * kVxSmallItems) return false;
  *slots = pow2AtLeast(static_cast<uint64_t>(numPts) * 2);
  *lds = static_cast<size_t>(*slots) * 8 + static_cast<size_t>(numPts) * (C + 1) * 4;
  return *lds <= 150 * 1024;
}

template <int CT>
int32_t launchSmall(const VoxelizeArgs& a, const VxGeom& g, uint32_t slots, size_t lds, hipStream_t stream) {
  static std::atomic<bool> granted{false};
  if (lds > 64 * 1024 && !granted.load(std::memory_order_acquire)) {
    D3D_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(&vxSmall<CT>), hipFuncAttributeMaxDynamicSharedMemorySize,
                                      150 * 1024));
    granted.store(true, std::memory_order_release);
  }
  const int64_t beyond = (static_cast<int64_t>(a.maxNumActOut) - a.numPts) * a.C;
  int64_t zeroing = beyond > 0 ? (beyond + kVxSmallThreads * 4 - 1) / (kVxSmallThreads * 4) : 0;
  if (zeroing > 512) zeroing = 512;
  hipLaunchKernelGGL(vxSmall<CT>, dim3(static_cast<unsigned>(1 + zeroing)), dim3(kVxSmallThreads), lds, stream, a.feats, a.batchIdx,
                     a.config, static_cast<int32_t>(a.numPts), a.C, g, slots - 1, a.maxNumActOut, a.outFeats, a.outCoors,
                     a.numActOut);
  D3D_HIP_CHECK(hipGetLastError());
  return D3D_OK;
}

template <int CT>
void launchWide(const VoxelizeArgs& a, const VxPlan& p, const VxGeom& g, char* ws, hipStream_t stream) {
  auto* table = reinterpret_cast<unsigned long long*>(ws);
  auto* records = reinterpret_cast<unsigned char*>(ws + p.records);
  auto* points = reinterpret_cast<uint2*>(ws + p.pointSlot);
  auto* states = reinterpret_cast<unsigned long long*>(ws + p.chunkBase);
  const int perRecord = vxRecordBytes(a.C) / 16;
  const int64_t pieces = a.numPts * perRecord, nFeats = static_cast<int64_t>(a.maxNumActOut) * a.C;
  int64_t blocks = (pieces + p.slots / 2 + kVxThreads * 4 - 1) / (kVxThreads * 4);
  if (blocks > 4096) blocks = 4096;
#define D3D_VX_CLEAR(PER)                                                                                                       \
  hipLaunchKernelGGL(vxClearWide<PER>, dim3(static_cast<unsigned>(blocks)), dim3(kVxThreads), 0, stream,                        \
                     reinterpret_cast<uint4*>(table), p.slots / 2, reinterpret_cast<uint4*>(records),                              \
                     static_cast<uint32_t>(pieces), a.outFeats, nFeats, states, p.nChunks)
  if (perRecord == 2) D3D_VX_CLEAR(2);
  else if (perRecord == 3) D3D_VX_CLEAR(3);
  else D3D_VX_CLEAR(4);
#undef D3D_VX_CLEAR
  hipLaunchKernelGGL(vxInsertWide<CT>, dim3(static_cast<unsigned>((a.numPts + kVxThreads - 1) / kVxThreads)), dim3(kVxThreads), 0,
                     stream, a.feats, a.batchIdx, a.config, static_cast<int32_t>(a.numPts), a.C, g, table, p.slots, records, points);
  hipLaunchKernelGGL((a.numPts <= kVxSmallChunks ? vxEmitWide<CT, 1> : vxEmitWide<CT, 2>), dim3(p.nChunks), dim3(kVxThreads), 0, stream, a.feats, static_cast<int32_t>(a.numPts), a.C, g,
                     records, points, states, a.maxNumActOut, a.outFeats, a.outCoors, a.numActOut);
}

}  // namespace

size_t voxelizeWorkspaceBytes(int64_t numPts, int64_t maxNumActOut, int64_t C) {
  return planVoxelize(numPts, maxNumActOut, C).total;
}

int32_t launchVoxelize(const VoxelizeArgs& a, hipStream_t stream) {
  const VxPlan p = planVoxelize(a.numPts, a.maxNumActOut, a.C);
  if (!a.workspace || a.workspaceBytes < p.total) {
    setError("SimpleMeanEncoder: workspace of %zu bytes, %zu needed", a.workspaceBytes, p.total);
    return D3D_ERR_WORKSPACE;
  }
  if (reinterpret_cast<uintptr_t>(a.workspace) % 16 != 0 || reinterpret_cast<uintptr_t>(a.outCoors) % 16 != 0) {
    setError("SimpleMeanEncoder: workspace and outCoors must start on 16-byte boundaries");
    return D3D_ERR_BAD_ARG;
  }
  const uint64_t cells = static_cast<uint64_t>(a.B) * a.Z * a.Y * a.X;
  if (cells >= 0xFFFFFFFFull) {
    setError("SimpleMeanEncoder: grid [%d, %d, %d, %d] has more cells than a 32-bit key can name", a.B, a.Z, a.Y, a.X);
    return D3D_ERR_UNSUPPORTED;
  }
  char* ws = static_cast<char*>(a.workspace);
  const VxGeom g{a.B, a.Z, a.Y, a.X};
  if (a.numPts > 0 && a.maxNumActOut > 0 && cells > 0) {
    uint32_t slots = 0;
    size_t lds = 0;
    if (smallFits(a.numPts, a.C, &slots, &lds)) {
      switch (a.C) {
        case 3: return launchSmall<3>(a, g, slots, lds, stream);
        case 4: return launchSmall<4>(a, g, slots, lds, stream);
        case 5: return launchSmall<5>(a, g, slots, lds, stream);
        default: return launchSmall<0>(a, g, slots, lds, stream);
      }
    }
    if (p.wide) {
      switch (a.C) {
        case 3: launchWide<3>(a, p, g, ws, stream); break;
        case 4: launchWide<4>(a, p, g, ws, stream); break;
        case 5: launchWide<5>(a, p, g, ws, stream); break;
        default: launchWide<0>(a, p, g, ws, stream);
      }
      D3D_HIP_CHECK(hipGetLastError());
      return D3D_OK;
    }
  }
  auto* table = reinterpret_cast<unsigned long long*>(ws + p.table);
  auto* pointSlot = reinterpret_cast<uint32_t*>(ws + p.pointSlot);
  auto* local = reinterpret_cast<uint32_t*>(ws + p.local);
  auto* chunkBase = reinterpret_cast<uint32_t*>(ws + p.chunkBase);
  auto* counts = reinterpret_cast<uint32_t*>(ws + p.counts);
  auto* ticket = reinterpret_cast<uint32_t*>(ws + p.ticket);
  const int64_t nFeats = static_cast<int64_t>(a.maxNumActOut) * a.C;
  if (p.wide) {  // nothing to insert: only the outputs' zeros (the plan has no table of bare keys)
    hipLaunchKernelGGL(vxReset, dim3(static_cast<unsigned>(nFeats < 1 ? 1 : (nFeats / kVxThreads > 4095 ? 4096 : nFeats / kVxThreads + 1))),
                       dim3(kVxThreads), 0, stream, nullptr, int64_t(0), a.outFeats, nFeats, nullptr, int64_t(0), a.numActOut);
    D3D_HIP_CHECK(hipGetLastError());
    return D3D_OK;
  }
  const int64_t resetItems = static_cast<int64_t>(p.slots) + nFeats;
  int64_t resetBlocks = (resetItems + kVxThreads - 1) / kVxThreads;
  if (resetBlocks > 4096) resetBlocks = 4096;
  hipLaunchKernelGGL(vxReset, dim3(static_cast<unsigned>(resetBlocks < 1 ? 1 : resetBlocks)), dim3(kVxThreads), 0, stream,
                     table, static_cast<int64_t>(p.slots), a.outFeats, nFeats, counts,
                     static_cast<int64_t>(a.maxNumActOut) + 1, a.numActOut);
  if (a.numPts > 0 && a.maxNumActOut > 0 && cells > 0) {
    const dim3 perPoint(static_cast<unsigned>((a.numPts + kVxThreads - 1) / kVxThreads));
    hipLaunchKernelGGL(vxInsert, perPoint, dim3(kVxThreads), 0, stream, a.feats, a.batchIdx, a.config,
                       static_cast<int32_t>(a.numPts), a.C, g, table, p.slots - 1, pointSlot);
    hipLaunchKernelGGL(vxRank, dim3(p.nChunks), dim3(kVxThreads), 0, stream, table, pointSlot,
                       static_cast<int32_t>(a.numPts), local, chunkBase, p.nChunks, ticket, a.numActOut, a.maxNumActOut);
    hipLaunchKernelGGL(vxAccumulate, perPoint, dim3(kVxThreads), 0, stream, a.feats, static_cast<int32_t>(a.numPts), a.C,
                       g, table, pointSlot, local, chunkBase, a.maxNumActOut, a.outFeats, counts, a.outCoors);
    int64_t meanBlocks = (nFeats + kVxThreads - 1) / kVxThreads;
    if (meanBlocks > 2048) meanBlocks = 2048;
    hipLaunchKernelGGL(vxMean, dim3(static_cast<unsigned>(meanBlocks)), dim3(kVxThreads), 0, stream, a.outFeats, counts,
                       a.numActOut, a.C);
  }
  D3D_HIP_CHECK(hipGetLastError());
  return D3D_OK;
}

}  // namespace d3d
