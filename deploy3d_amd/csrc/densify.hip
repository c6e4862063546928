// Sparse rows -> dense bird's-eye-view feature map.
//
// The dense map is [B, C, Z, Y, X] (handed on as [B, C*Z, Y, X]); voxel row i
// with coordinate (b, z, y, x) fills out[b, :, z, y, x] and every other cell is
// zero (reference: kernel::densify and the memset before it,
// trt/spconv/bev_densify_trt.cu:22-35, :160-174).
//
// The reference clears the map and then scatters one channel at a time, so a
// row of C values lands in C different cache lines.  Here the map is produced
// output-stationary instead: a cell -> row table is built first (4 bytes per
// cell), then every workgroup owns 64 consecutive cells of one (b, z) plane,
// pulls the rows of its occupied cells through LDS and writes whole runs of
// 64 cells per channel, zeros included.  Each output byte is written exactly
// once and no clearing pass is needed.
//
// The table is not cleared either: an entry counts only if it names a live row
// whose coordinate IS the cell, so whatever the workspace held before is told
// apart from an entry by one 16-byte load (two launches instead of three:
// 11.3 -> 10.2 us per call in a graph of calls, for 38 000 rows of 128 fp16
// channels into [1, 256, 180, 180]: 26.3 MB, which a large copy moves in 5.7).
#include "common.h"
#include "conv_kernels.h"
#include "densify_grid.h"

namespace d3d {
namespace {

constexpr int kTile = kDzTile, kChunkBytes = kDzChunkBytes;
constexpr int kPitch = kChunkBytes + 4;  // LDS bytes per cell: an odd number of dwords

struct DzGrid {
  int B, Z, Y, X;
};

__device__ __forceinline__ bool dzCellOf(const int4& c, const DzGrid& g, int64_t* cell) {
  if (static_cast<unsigned>(c.x) >= static_cast<unsigned>(g.B) || static_cast<unsigned>(c.y) >= static_cast<unsigned>(g.Z) ||
      static_cast<unsigned>(c.z) >= static_cast<unsigned>(g.Y) || static_cast<unsigned>(c.w) >= static_cast<unsigned>(g.X))
    return false;
  *cell = ((static_cast<int64_t>(c.x) * g.Z + c.y) * g.Y + c.z) * g.X + c.w;
  return true;
}

// The row a table entry stands for: a live row at this very cell, else -1.
__device__ __forceinline__ int32_t dzRowAt(int32_t entry, int64_t cell, const int32_t* __restrict__ coors, int32_t n, const DzGrid& g) {
  if (static_cast<unsigned>(entry) >= static_cast<unsigned>(n)) return -1;
  int64_t at;
  return dzCellOf(reinterpret_cast<const int4*>(coors)[entry], g, &at) && at == cell ? entry : -1;
}

__device__ __forceinline__ int32_t dzLive(const int32_t* numAct, int32_t cap) { return min(max(*numAct, 0), cap); }

// The highest row wins a cell named twice, which is what a serial pass over
// the rows leaves behind.  Rows outside the grid are dropped.  A row replaces
// what the table held unless that is a higher row of the same cell.
__global__ __launch_bounds__(256) void dzMapRows(const int32_t* __restrict__ coors, const int32_t* __restrict__ numAct,
                                                 int32_t cap, DzGrid g, int32_t* __restrict__ map) {
  const int32_t n = dzLive(numAct, cap);
  const int32_t i = blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  int64_t cell;
  if (!dzCellOf(reinterpret_cast<const int4*>(coors)[i], g, &cell)) return;
  int32_t seen = map[cell];
  while (dzRowAt(seen, cell, coors, n, g) < i) {   // every failed exchange met another row of this cell: at most n turns
    const int32_t old = atomicCAS(map + cell, seen, i);
    if (old == seen) break;
    seen = old;
  }
}

// grid: (tiles of a plane, B*Z planes, channel chunks).  E = bytes per element,
// PACK = cells written by one store (PACK*E == 16 or 4, or PACK == 1), VEC = rows are
// fetched in 16-byte pieces.
// PACK*E == 16: a thread reads the 4/E channels of a dword for PACK cells and stores them channel by channel, 16 bytes each:
// a quarter of the LDS reads and of the stores of an element at a time.
template <int E, int PACK, bool VEC>
__global__ __launch_bounds__(256) void dzGather(const uint8_t* __restrict__ feats, const int32_t* __restrict__ map,
                                                const int32_t* __restrict__ coors, const int32_t* __restrict__ numAct,
                                                int32_t cap, DzGrid g, uint8_t* __restrict__ out, int C, int64_t YX, uint32_t tiles, uint32_t pieces, int xcdShift) {
  __shared__ int32_t rows[kTile];
  __shared__ __attribute__((aligned(16))) uint8_t tile[kTile * kPitch];

  const int t = threadIdx.x;
  uint32_t tileAt = blockIdx.x, planeAt = blockIdx.y, chunkAt = blockIdx.z;
  if (pieces) {   // one-dimensional: XCD x takes the x-th contiguous part, so that lines two tiles share are whole in one L2
    const uint32_t piece = (blockIdx.x & ((1u << xcdShift) - 1u)) * (gridDim.x >> xcdShift) + (blockIdx.x >> xcdShift);
    if (piece >= pieces) return;
    tileAt = piece % tiles;
    planeAt = piece / tiles % (g.B * g.Z);
    chunkAt = piece / tiles / (g.B * g.Z);
  }
  const int64_t p0 = static_cast<int64_t>(tileAt) * kTile;
  const int plane = planeAt;
  const int Z = g.Z, b = plane / Z, z = plane % Z;
  const int c0 = chunkAt * (kChunkBytes / E);             // first channel of this chunk
  const int cc = min(kChunkBytes / E, C - c0);            // channels in this chunk
  const int ccBytes = cc * E;
  const size_t rowBytes = static_cast<size_t>(C) * E;

  if (t < kTile) {
    const int64_t cell = static_cast<int64_t>(plane) * YX + p0 + t;
    rows[t] = p0 + t < YX ? dzRowAt(map[cell], cell, coors, dzLive(numAct, cap), g) : -1;
  }
  __syncthreads();

  if constexpr (VEC) {
    // 8 lanes x 16 bytes per cell, 32 cells per sweep
    for (int u = t; u < kTile * (kChunkBytes / 16); u += 256) {
      const int cell = u / (kChunkBytes / 16), q = u % (kChunkBytes / 16);
      if (q * 16 >= ccBytes) continue;
      const int r = rows[cell];
      uint4 v = make_uint4(0, 0, 0, 0);
      if (r >= 0) v = *reinterpret_cast<const uint4*>(feats + r * rowBytes + static_cast<size_t>(c0) * E + q * 16);
      uint32_t* dst = reinterpret_cast<uint32_t*>(tile + cell * kPitch + q * 16);
      dst[0] = v.x;
      dst[1] = v.y;
      dst[2] = v.z;
      dst[3] = v.w;
    }
  } else {
    for (int u = t; u < kTile * ccBytes; u += 256) {
      const int cell = u / ccBytes, q = u % ccBytes;
      const int r = rows[cell];
      tile[cell * kPitch + q] = r >= 0 ? feats[r * rowBytes + static_cast<size_t>(c0) * E + q] : uint8_t(0);
    }
  }
  __syncthreads();

  constexpr int kGroups = kTile / PACK;  // stores per channel
  if constexpr (PACK * E == 16) {
    constexpr int CH = 4 / E;            // channels of a dword
    for (int u = t; u < cc / CH * kGroups; u += 256) {
      const int ch = u / kGroups * CH, cell0 = (u % kGroups) * PACK;
      const int64_t p = p0 + cell0;
      if (p >= YX) continue;
      uint32_t in[PACK];
#pragma unroll
      for (int e = 0; e < PACK; ++e) in[e] = *reinterpret_cast<const uint32_t*>(tile + (cell0 + e) * kPitch + ch * E);
      const size_t at = (((static_cast<size_t>(b) * C + c0 + ch) * Z + z) * YX + p) * E, step = static_cast<size_t>(Z) * YX * E;
#pragma unroll
      for (int k = 0; k < CH; ++k) {
        uint32_t w[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          if constexpr (E == 4) {
            w[q] = in[q];
          } else if constexpr (E == 2) {   // halves k of cells 2q and 2q + 1
            w[q] = __builtin_amdgcn_perm(in[2 * q + 1], in[2 * q], k ? 0x07060302u : 0x05040100u);
          } else {                         // bytes k of cells 4q .. 4q + 3
            const uint32_t pick = 0x0400u + 0x0101u * k;
            w[q] = __builtin_amdgcn_perm(__builtin_amdgcn_perm(in[4 * q + 3], in[4 * q + 2], pick),
                                         __builtin_amdgcn_perm(in[4 * q + 1], in[4 * q], pick), 0x05040100u);
          }
        }
        *reinterpret_cast<uint4*>(out + at + k * step) = make_uint4(w[0], w[1], w[2], w[3]);
      }
    }
    return;
  }
  for (int u = t; u < cc * kGroups; u += 256) {
    const int ch = u / kGroups, cell0 = (u % kGroups) * PACK;
    const int64_t p = p0 + cell0;
    if (p >= YX) continue;
    const size_t at = (((static_cast<size_t>(b) * C + c0 + ch) * Z + z) * YX + p) * E;
    const uint8_t* src = tile + cell0 * kPitch + ch * E;
    if constexpr (E == 4) {
      *reinterpret_cast<uint32_t*>(out + at) = *reinterpret_cast<const uint32_t*>(src);
    } else if constexpr (E == 2) {
      if constexpr (PACK == 2) {
        const uint32_t lo = *reinterpret_cast<const uint16_t*>(src);
        const uint32_t hi = *reinterpret_cast<const uint16_t*>(src + kPitch);
        *reinterpret_cast<uint32_t*>(out + at) = lo | (hi << 16);
      } else {
        *reinterpret_cast<uint16_t*>(out + at) = *reinterpret_cast<const uint16_t*>(src);
      }
    } else {
      if constexpr (PACK == 4) {
        const uint32_t v = uint32_t(src[0]) | (uint32_t(src[kPitch]) << 8) | (uint32_t(src[2 * kPitch]) << 16) |
                           (uint32_t(src[3 * kPitch]) << 24);
        *reinterpret_cast<uint32_t*>(out + at) = v;
      } else {
        out[at] = src[0];
      }
    }
  }
}

template <int E>
void launchGather(const DensifyArgs& a, const int32_t* map, hipStream_t stream) {
  const int xcdShift = convk::chipLayout().xcdShift;
  const int64_t yx = static_cast<int64_t>(a.Y) * a.X;
  const DensifyGrid dg = densifyGrid(yx, static_cast<int64_t>(a.B) * a.Z, a.C, E, xcdShift);
  const dim3 grid(dg.x, dg.y, dg.z);
  const bool vec = (static_cast<size_t>(a.C) * E) % 16 == 0 && reinterpret_cast<uintptr_t>(a.feats) % 16 == 0;
  const bool wide = yx % (16 / E) == 0 && reinterpret_cast<uintptr_t>(a.out) % 16 == 0 && a.C * E % 4 == 0;
  constexpr int kPack = 4 / E;
  const bool pack = kPack > 1 && yx % kPack == 0 && reinterpret_cast<uintptr_t>(a.out) % 4 == 0;
  const DzGrid g{a.B, a.Z, a.Y, a.X};
  const uint8_t* f = static_cast<const uint8_t*>(a.feats);
  uint8_t* o = static_cast<uint8_t*>(a.out);
#define D3D_DZ(P, V) hipLaunchKernelGGL((dzGather<E, P, V>), grid, dim3(256), 0, stream, f, map, a.coors, a.numAct, a.cap, g, o, a.C, yx, static_cast<uint32_t>((yx + kTile - 1) / kTile), dg.pieces, xcdShift)
  if (wide) {
    if (vec) D3D_DZ(16 / E, true); else D3D_DZ(16 / E, false);
  } else if (pack) {
    if (vec) D3D_DZ(kPack, true); else D3D_DZ(kPack, false);
  } else {
    if (vec) D3D_DZ(1, true); else D3D_DZ(1, false);
  }
#undef D3D_DZ
}

}  // namespace

size_t densifyWorkspaceBytes(int64_t B, int64_t Z, int64_t Y, int64_t X) {
  return static_cast<size_t>(B * Z * Y * X) * sizeof(int32_t);
}

int32_t launchDensify(const DensifyArgs& a, hipStream_t stream) {
  const int64_t cells = static_cast<int64_t>(a.B) * a.Z * a.Y * a.X;
  if (cells == 0 || a.C == 0) return D3D_OK;  // nothing to write
  const int64_t planes = static_cast<int64_t>(a.B) * a.Z;
  const int E = a.elemBytes;
  const int64_t chunks = (static_cast<int64_t>(a.C) * E + kChunkBytes - 1) / kChunkBytes;
  if (E != 1 && E != 2 && E != 4) {
    setError("BEVDensify: elements of %d bytes not implemented", E);
    return D3D_ERR_UNSUPPORTED;
  }
  if (planes > 65535 || chunks > 65535 || cells >= (int64_t(1) << 31)) {
    setError("BEVDensify: grid [%d, %d, %d, %d] x %d channels exceeds the launch limits", a.B, a.Z, a.Y, a.X, a.C);
    return D3D_ERR_BAD_ARG;
  }
  if (a.workspaceBytes < static_cast<size_t>(cells) * 4 || !a.workspace) {
    setError("BEVDensify: workspace of %zu bytes, %zu needed", a.workspaceBytes, static_cast<size_t>(cells) * 4);
    return D3D_ERR_WORKSPACE;
  }
  if (reinterpret_cast<uintptr_t>(a.coors) % 16 != 0) {
    setError("BEVDensify: coordinate rows must start on a 16-byte boundary");
    return D3D_ERR_BAD_ARG;
  }
  int32_t* map = static_cast<int32_t*>(a.workspace);
  if (a.cap > 0)
    hipLaunchKernelGGL(dzMapRows, dim3(static_cast<unsigned>((a.cap + 255) / 256)), dim3(256), 0, stream, a.coors,
                       a.numAct, a.cap, DzGrid{a.B, a.Z, a.Y, a.X}, map);
  if (E == 4) launchGather<4>(a, map, stream);
  else if (E == 2) launchGather<2>(a, map, stream);
  else launchGather<1>(a, map, stream);
  D3D_HIP_CHECK(hipGetLastError());
  return D3D_OK;
}

}  // namespace d3d
