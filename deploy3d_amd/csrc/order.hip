// Rows of a neighbour table in the order of their taps (inverse convolutions): see orderRows.
#include "conv_kernels.h"

namespace d3d {
namespace {

using namespace convk;

// Class of a tap mask, 0 .. 62.  Rows of an inverse convolution have as many different masks as the stride has positions
// (eight at stride 2: 1, 2, 4 or 8 of 27 taps) and those at the grid's edges; the factor keeps those of the usual kernels
// (3x3x3 at strides 2 and 3, 2x2x2, 3x1x3, 3x3, 4x4) apart.  Masks that share a class cost time, not results.
__host__ __device__ inline uint32_t tapClass(uint32_t mask) { return (mask * 0x2265B1F5u >> 26) % 63u; }

// An output row of an inverse convolution has the taps its position in the stride allows, 27/8 of 27 on average at stride 2,
// and its neighbours in memory have the others: every tile multiplied every tap.  Here the rows of a window are sorted by
// class, stably, so the result does not vary from run to run.  One workgroup a window: a thread holds the table entries of
// two rows in registers, ranks them among the rows of their class (wavefront by wavefront with ballots, then one scan over
// classes and wavefronts), and the columns go back through LDS, coalesced.
// Windows of 512 rows: what a workgroup reads and writes, through one CU, is the time.  128 000 rows (14 MB in, 14 MB out) and
// 40 000 take 16 and 15 us in windows of 2048, 11 and 10 in 1024, 10 and 7.6 in 512, while 128-row tiles hold 25, 35 and 54 % of
// the taps and 16-row groups 14, 15 and 17: fp32 64 -> 32 behind it 46, 45.5 and 50.5 us (119 unsorted), 32 -> 16 16.7, 16.2 and
// 15.4 (27).  Encoder-decoder of 40 000 voxels in fp32 797 -> 751, 740 and 734 us.  Which
// layers gain by it: MMPlugin::ordersRows.
// Rows past the live ones keep to the end of the last window that has live rows; windows behind it hold no neighbours and
// are not read.
template <int MAXTAPS>
__global__ void __launch_bounds__(kOrderWindow / 2)
orderRows(int32_t* __restrict__ nbr, int kVol, int64_t outRows, const int32_t* __restrict__ numActOut, RowOrder out) {
  constexpr int W = kOrderWindow, PER = 2, THREADS = W / PER, WAVES = THREADS / 64, BATCH = 14;
  static_assert(W % 128 == 0 && 2 * BATCH * W * 4 <= 64 * 1024, "a thread holds rows 2 * tid and 2 * tid + 1, and scans one of 64 * WAVES places");
  __shared__ __attribute__((aligned(16))) int32_t column[BATCH][W];
  __shared__ uint32_t count[64 * WAVES];                  // rows of (class, wavefront); then the places before them
  __shared__ uint32_t waveSum[WAVES];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int64_t w0 = static_cast<int64_t>(blockIdx.x) * W;
  int64_t live = numActOut ? *numActOut : outRows;
  live = live < 0 ? 0 : (live > outRows ? outRows : live);
  if (blockIdx.x == gridDim.x - 1 && tid < 8) out.masks[static_cast<int64_t>(gridDim.x) * (W / 64) + tid] = 0;  // tiles are read whole
  if (w0 >= live) {                                       // workgroup-uniform
    for (int r = tid; r < W; r += THREADS) {
      if (w0 + r >= outRows) break;
      out.rows[w0 + r] = static_cast<int32_t>(w0 + r);
      for (int t = 0; t < kVol; ++t) nbr[static_cast<int64_t>(t) * outRows + w0 + r] = -1;
    }
    if (tid < W / 64) out.masks[w0 / 64 + tid] = 0;
    return;
  }

  const uint32_t at = static_cast<uint32_t>(w0) + 2 * tid, rows = static_cast<uint32_t>(outRows);
  const bool whole = w0 + W <= outRows;                   // workgroup-uniform
  const __amdgpu_buffer_rsrc_t table = makeRawBuffer(nbr, static_cast<uint32_t>(kVol) * rows * 4u);
  // rows past the table repeat its last one and are cut below (a pair that starts there ends in the next tap's column or, four
  // bytes behind the table, in `out`)
  const uint32_t from = at < rows ? at : rows - 1u;
  u32x2 entry[MAXTAPS];
#pragma unroll
  for (int t = 0; t < MAXTAPS; ++t)
    entry[t] = t < kVol ? __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(table, from * 4u, static_cast<int>(t * rows * 4u), 0)) : u32x2{~0u, ~0u};
  count[tid] = 0;
  __syncthreads();
  uint32_t mask[PER], cls[PER];
#pragma unroll
  for (int p = 0; p < PER; ++p) {
    mask[p] = 0;
    const bool there = whole || at + p < rows;
#pragma unroll
    for (int t = 0; t < MAXTAPS; ++t) {
      if (!there) entry[t][p] = ~0u;
      mask[p] |= (~entry[t][p] >> 31) << t;
    }
    cls[p] = at + p < live ? tapClass(mask[p]) : 63u;
  }
  // a row's place among the rows of its class in the wavefront: those of lower lanes, both rows of a lane in turn
  uint32_t rank[PER];
  unsigned long long same[PER][PER];                      // [p][q]: lanes whose row q has the class of this lane's row p
#pragma unroll
  for (int p = 0; p < PER; ++p)
#pragma unroll
    for (int q = 0; q < PER; ++q) same[p][q] = ~0ull;
#pragma unroll
  for (int b = 0; b < 6; ++b)
#pragma unroll
    for (int q = 0; q < PER; ++q) {
      const unsigned long long ones = __ballot((cls[q] >> b) & 1);
#pragma unroll
      for (int p = 0; p < PER; ++p) same[p][q] &= (cls[p] >> b) & 1 ? ones : ~ones;
    }
  auto below = [](unsigned long long m, uint32_t add) __attribute__((always_inline)) {
    return __builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(m >> 32), __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(m), add));
  };
#pragma unroll
  for (int p = 0; p < PER; ++p) {
    rank[p] = below(same[p][1], below(same[p][0], 0u)) + (p == 1 && cls[0] == cls[1] ? 1u : 0u);
    if (rank[p] == 0) count[cls[p] * WAVES + wave] = __builtin_popcountll(same[p][0]) + __builtin_popcountll(same[p][1]);
  }
  __syncthreads();
  {  // exclusive scan over (class, wavefront), one entry a thread
    const uint32_t mine = count[tid];
    uint32_t incl = mine;
#pragma unroll
    for (int d = 1; d < 64; d *= 2) {
      const uint32_t v = __shfl_up(incl, d);
      if (lane >= d) incl += v;
    }
    if (lane == 63) waveSum[wave] = incl;
    __syncthreads();
    uint32_t before = 0;
#pragma unroll
    for (int i = 0; i < WAVES; ++i) before += i < wave ? waveSum[i] : 0u;
    count[tid] = before + incl - mine;
  }
  __syncthreads();
  uint32_t place[PER];
#pragma unroll
  for (int p = 0; p < PER; ++p) {
    place[p] = count[cls[p] * WAVES + wave] + rank[p];
    column[0][place[p]] = static_cast<int32_t>(at + p);
    column[1][place[p]] = static_cast<int32_t>(mask[p]);
  }
  __syncthreads();
  {
    const u32x2 r = *reinterpret_cast<const u32x2*>(&column[0][2 * tid]), m2 = *reinterpret_cast<const u32x2*>(&column[1][2 * tid]);
#pragma unroll
    for (int p = 0; p < PER; ++p)
      if (at + p < rows) out.rows[at + p] = static_cast<int32_t>(r[p]);
    uint32_t m = m2[0] | m2[1];                           // 32 lanes hold a 64-row tile
#pragma unroll
    for (int d = 1; d < 32; d *= 2) m |= __shfl_xor(m, d);
    if ((lane & 31) == 0) out.masks[at / 64] = m;
  }
#pragma unroll
  for (int t0 = 0; t0 < MAXTAPS; t0 += BATCH) {
    if (t0 >= kVol) break;
    __syncthreads();
#pragma unroll
    for (int q = 0; q < BATCH; ++q)
#pragma unroll
      for (int p = 0; p < PER; ++p)
        if (t0 + q < MAXTAPS) column[q][place[p]] = static_cast<int32_t>(entry[t0 + q < MAXTAPS ? t0 + q : 0][p]);
    __syncthreads();
#pragma unroll
    for (int q = 0; q < BATCH; ++q) {
      if (t0 + q >= kVol) break;
      const u32x2 v = *reinterpret_cast<const u32x2*>(&column[q][2 * tid]);
      const int tap = static_cast<int>((t0 + q) * rows * 4u);
      if (whole) {
        __builtin_amdgcn_raw_buffer_store_b64(v, table, at * 4u, tap, 0);
      } else {
        if (at < rows) __builtin_amdgcn_raw_buffer_store_b32(v[0], table, at * 4u, tap, 0);
        if (at + 1 < rows) __builtin_amdgcn_raw_buffer_store_b32(v[1], table, at * 4u + 4u, tap, 0);
      }
    }
  }
}

int64_t orderWindows(int64_t outRows) { return (outRows + kOrderWindow - 1) / kOrderWindow; }

}  // namespace

size_t orderRowsBytes(int64_t outRows) {
  return static_cast<size_t>((outRows + 1) / 2 * 2) * sizeof(int32_t) + static_cast<size_t>(orderWindows(outRows) * (kOrderWindow / 64) + 8) * 8;
}

RowOrder orderRowsAt(void* base, int64_t outRows) {
  int32_t* const rows = static_cast<int32_t*>(base);
  return {rows, reinterpret_cast<unsigned long long*>(rows + (outRows + 1) / 2 * 2)};
}

int32_t launchOrderRows(int32_t* nbr, int kVol, int64_t outRows, const int32_t* numActOut, const RowOrder& out, hipStream_t stream) {
  if (outRows <= 0) return D3D_OK;
  auto* const kernel = kVol <= 27 ? &orderRows<27> : &orderRows<32>;
  hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(orderWindows(outRows))), dim3(kOrderWindow / 2), 0, stream, nbr, kVol, outRows,
                     numActOut, out);
  D3D_HIP_CHECK(hipGetLastError());
  return D3D_OK;
}

}  // namespace d3d
