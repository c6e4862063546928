// MFMA convolution for 32 -> 32 channels in two-byte types: weights of every tap resident in LDS, wavefronts that run
// alone.
//
// Same mathematics, row layout and table reads as convPipe (conv_pipe.h).  A 32-channel step is short - 8 MFMAs, four
// gathers of 16 rows, ten LDS reads - so in convPipe the barrier of every step and the weight slice that all wavefronts
// fetch for it weigh as much as the step itself, and 512-row tiles leave the busiest CU a third more rows than the
// average.  Here all 27 taps of weights (54 KB) stay in LDS, the twelve wavefronts of a CU share them and nothing else,
// and each walks its own 64-row tiles: indices four steps ahead, rows two steps ahead, across tiles.
// What bounds it: 10 KB through LDS per step (gathered rows in and out, weights) at 128 bytes per clock, 80 of the 110
// clocks that a step takes per CU; a gather moves 64 bytes per clock into a CU whether its rows are present or not.
// Rows gathered straight into the MFMA's register layout avoid the LDS round trip, but a load whose neighbouring lanes
// read different rows takes up to three times as long: 46 us where this takes 36.
// Measured (convPipe before): 349 000 rows 36 us (38), 1.35 million rows 149 us (156), 26 000 rows 10 us (17).
#pragma once
#include "conv_pipe.h"

namespace d3d {
namespace convk {

template <class T, int COUT, int WAVES>
__global__ void __launch_bounds__(64 * WAVES)
convSolo(const T* __restrict__ in, T* __restrict__ out, const T* __restrict__ wf, const float* __restrict__ bias,
         const int32_t* __restrict__ nbr, uint32_t nbrPitch, int tapMirror, const unsigned long long* __restrict__ tileMasks,
         int kVol, int64_t inRows, int64_t outRows, int relu, int tiles, int perBlock, int xcdShift,
         const int32_t* __restrict__ numActOut) {
  constexpr int MT = 4, NT = COUT / 16, WM = 16 * MT;
  constexpr int CH = 4, RPI = 16;                    // 16-byte chunks of a 64-byte row; rows one gather instruction covers
  constexpr int SLOTS = WM * CH;                     // 16-byte slots of one stage
  constexpr int WCH = 32 * COUT * 2 / 16;            // 16-byte chunks of one tap's weights
  constexpr int NI = 3;                              // index ring depth (steps)
  static_assert(sizeof(T) == 2 && NT == 2, "32 -> 32 channels");

  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r16 = lane & 15, kgrp = lane >> 4;
  u32x4* const wLds = reinterpret_cast<u32x4*>(smem);                                             // [kVol][WCH]
  u32x4* const stage = wLds + kVol * WCH + wave * 2 * SLOTS;                                      // [2][SLOTS]
  int32_t* const idxLds = reinterpret_cast<int32_t*>(wLds + kVol * WCH + WAVES * 2 * SLOTS) + wave * NI * WM;  // [NI][WM]
  for (int e = tid; e < kVol * WCH; e += 64 * WAVES) wLds[e] = reinterpret_cast<const u32x4*>(wf)[e];
  __syncthreads();

  const TileOrder order(tiles, static_cast<int>((liveOutRows(numActOut, outRows) + WM - 1) / WM), xcdShift,
                        blockIdx.x & ((1 << xcdShift) - 1));
  const int firstLocal = (blockIdx.x >> xcdShift) * perBlock + wave, strideLocal = (gridDim.x >> xcdShift) * perBlock;
  const int nMine = wave < perBlock && firstLocal < order.count() ? (order.count() - 1 - firstLocal) / strideLocal + 1 : 0;
  if (nMine <= 0) return;
  auto tileAt = [&](int pos) __attribute__((always_inline)) {
    return __builtin_amdgcn_readfirstlane(order.tile(firstLocal + pos * strideLocal));
  };
  const uint32_t allTaps = kVol >= 32 ? ~0u : (1u << kVol) - 1u;
  auto maskAt = [&](int pos) __attribute__((always_inline)) -> uint32_t {
    if (pos >= nMine) return 0u;
    if (!order.live(firstLocal + pos * strideLocal)) return 1u;   // no live row: one step of absent neighbours
    uint32_t m = allTaps;
    if (tileMasks) m &= static_cast<uint32_t>(tileMasks[tileAt(pos)]);
    m = __builtin_amdgcn_readfirstlane(m);
    return m ? m : 1u;
  };

  const __amdgpu_buffer_rsrc_t inBuf = makeRawBuffer(in, static_cast<uint32_t>(inRows * 64));
  const __amdgpu_buffer_rsrc_t nbrBuf = makeRawBuffer(nbr, static_cast<uint32_t>(kVol) * nbrPitch * 4u);
  const uint32_t chunkOff = static_cast<uint32_t>(((lane % CH) ^ stageSwizzle<CH>(lane / CH)) * 16);
  // ring position `lane` holds the index of tile row (lane % 4) * 16 + lane / 4: a lane's four gathers read 16 bytes
  const uint32_t idxOff = static_cast<uint32_t>(((lane % MT) * RPI + lane / MT) * 4);
  const int readAt = r16 * CH + (kgrp ^ stageSwizzle<CH>(r16));   // row fragment of group m: + m * 16 * CH

  // ---- the walk over (tile, tap): see convPipe ----
  constexpr uint32_t kLastOfTile = 1u << 31;
  int walkPos = 0;
  uint32_t walkRem = maskAt(0), walkTaps = maskAt(1), walkTap = 0;
  uint32_t rowBytes = static_cast<uint32_t>(tileAt(0)) * (WM * 4u);
  auto loadIndex = [&](int slot) __attribute__((always_inline)) -> uint32_t {
    if (walkRem == 0 && walkPos + 1 < nMine) {
      ++walkPos;
      walkRem = walkTaps;
      walkTaps = maskAt(walkPos + 1);
      rowBytes = static_cast<uint32_t>(tileAt(walkPos)) * (WM * 4u);
    }
    if (walkRem) {
      walkTap = static_cast<uint32_t>(__builtin_ctz(walkRem));
      walkRem &= walkRem - 1;
    }
    const uint32_t tapRow = tapMirror ? static_cast<uint32_t>(kVol) - 1u - walkTap : walkTap;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(nbrBuf, (LdsVoidPtr)(idxLds + slot * WM), 4, tapRow * nbrPitch * 4u + rowBytes + idxOff, 0, 0, 0);
    return walkTap | (walkRem == 0 ? kLastOfTile : 0u);
  };
  auto gather = [&](int j, int32_t idx, int slot) __attribute__((always_inline)) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(inBuf, (LdsVoidPtr)(stage + slot * SLOTS + j * 64), 16,
                                             (static_cast<uint32_t>(idx) << 6) + chunkOff, 0, 0, 0);
  };

  float4v acc[MT][NT];
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int n = 0; n < NT; ++n) acc[m][n] = float4v{0.f, 0.f, 0.f, 0.f};

  auto storeTile = [&](int pos) __attribute__((always_inline)) {
    const int64_t row0 = static_cast<int64_t>(tileAt(pos)) * WM;
    const int col0 = kgrp * 4;
    const float4v b0 = bias ? *reinterpret_cast<const float4v*>(bias + col0) : float4v{0.f, 0.f, 0.f, 0.f};
    const float4v b1 = bias ? *reinterpret_cast<const float4v*>(bias + col0 + 16) : float4v{0.f, 0.f, 0.f, 0.f};
    const int outCol = (kgrp & 1) * 16 + (kgrp >> 1) * 8;
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      T p0[4], p1[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        float v0 = acc[m][0][j] + b0[j], v1 = acc[m][1][j] + b1[j];
        if (relu) {
          v0 = v0 > 0.f ? v0 : 0.f;
          v1 = v1 > 0.f ? v1 : 0.f;
        }
        p0[j] = static_cast<T>(v0);
        p1[j] = static_cast<T>(v1);
      }
      acc[m][0] = float4v{0.f, 0.f, 0.f, 0.f};
      acc[m][1] = float4v{0.f, 0.f, 0.f, 0.f};
      const u32x2 a = __builtin_bit_cast(u32x2, p0), c = __builtin_bit_cast(u32x2, p1);
      const auto s0 = __builtin_amdgcn_permlane16_swap(a[0], c[0], false, false);
      const auto s1 = __builtin_amdgcn_permlane16_swap(a[1], c[1], false, false);
      const u32x4 line = {s0[0], s1[0], s0[1], s1[1]};
      const int64_t row = row0 + m * 16 + r16;
      if (row < outRows) *reinterpret_cast<u32x4*>(out + static_cast<size_t>(row) * COUT + outCol) = line;
    }
  };

  // ---- prologue: indices of steps 0..2, rows of steps 0 and 1, index of step 3 ----
  uint32_t ids[5];
  ids[0] = loadIndex(0);
  ids[1] = loadIndex(1);
  ids[2] = loadIndex(2);
  waitVmcnt<0>();
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    const int4v ix = *reinterpret_cast<const int4v*>(idxLds + t * WM + (lane / CH) * MT);
#pragma unroll
    for (int j = 0; j < MT; ++j) gather(j, ix[j], t);
  }
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  ids[3] = loadIndex(0);
  waitVmcnt<0>();

  int mulPos = 0;
  int ixRead = 2, ixWrite = 1;                       // ring slots of step a+2's indices / for step a+4's
  auto step = [&](auto slotTag) __attribute__((always_inline)) -> bool {
    constexpr int SLOT = decltype(slotTag)::value;
    // in flight behind what this step needs: the index of step a+3 and the four gathers of step a+1
    waitVmcnt<1 + MT>();
    const int4v ix = *reinterpret_cast<const int4v*>(idxLds + ixRead * WM + (lane / CH) * MT);
    u32x4 rows[MT], wts[NT];
    const u32x4* wTap = wLds + (ids[0] & ~kLastOfTile) * WCH + lane;
#pragma unroll
    for (int n = 0; n < NT; ++n) wts[n] = wTap[n * 64];
#pragma unroll
    for (int m = 0; m < MT; ++m) rows[m] = stage[SLOT * SLOTS + readAt + m * 16 * CH];
    ids[4] = loadIndex(ixWrite);
    ixRead = ixRead == NI - 1 ? 0 : ixRead + 1;
    ixWrite = ixWrite == NI - 1 ? 0 : ixWrite + 1;
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // the stage has been read: it may be refilled
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      gather(m, ix[m], SLOT);
#pragma unroll
      for (int n = 0; n < NT; ++n) acc[m][n] = Mfma<T>::k32(wts[n], rows[m], acc[m][n]);
    }
    const bool last = (ids[0] & kLastOfTile) != 0;
#pragma unroll
    for (int t = 0; t < 4; ++t) ids[t] = ids[t + 1];
    return last;
  };
  for (;;) {
    if (step(std::integral_constant<int, 0>{})) {
      storeTile(mulPos);
      if (++mulPos >= nMine) break;
    }
    if (step(std::integral_constant<int, 1>{})) {
      storeTile(mulPos);
      if (++mulPos >= nMine) break;
    }
  }
  waitVmcnt<0>();
}

// Twelve wavefronts of 64 rows per CU: 54 KB of weights, 8 KB of stage and 768 bytes of indices each.
template <class T>
int32_t launchSolo(const ConvArgs& a, hipStream_t stream) {
  constexpr int WAVES = 12, COUT = 32, WM = 64;
  const size_t lds = static_cast<size_t>(a.kVol) * (32 * COUT * 2) + static_cast<size_t>(WAVES) * (2 * WM * 64 + 3 * WM * 4);
  const int64_t pitch = a.nbrPitch > 0 ? a.nbrPitch : a.outRows;
  if (a.cin != 32 || a.cout != COUT || a.kVol > 32 || lds > kLdsLimit) return D3D_ERR_UNSUPPORTED;
  if (static_cast<uint64_t>(a.inRows) * 64 >= 0xFFFF0000ull ||
      static_cast<uint64_t>(a.kVol) * static_cast<uint64_t>(pitch) * 4 >= 0xFFFF0000ull ||
      static_cast<uint64_t>(a.outRows) + WM >= 0x3FFFFFFFull)
    return D3D_ERR_UNSUPPORTED;                         // 32-bit buffer offsets
  static std::atomic<size_t> granted{64 * 1024};
  const int32_t rc = grantLds(&convSolo<T, COUT, WAVES>, lds, &granted);
  if (rc != D3D_OK) return rc;
  const int tiles = static_cast<int>((a.outRows + WM - 1) / WM);
  const ChipLayout chip = chipLayout();
  const int nXcd = 1 << chip.xcdShift;
  const int maxBlocks = chip.cus / nXcd * nXcd;
  const int blocks = tiles < maxBlocks ? (tiles + nXcd - 1) / nXcd * nXcd : maxBlocks;
  int perBlock = (tiles + blocks - 1) / blocks;         // few tiles spread over the CUs before they share one
  if (perBlock > WAVES) perBlock = WAVES;
  hipLaunchKernelGGL((convSolo<T, COUT, WAVES>), dim3(static_cast<unsigned>(blocks)), dim3(64 * WAVES), lds, stream,
                     static_cast<const T*>(a.in), static_cast<T*>(a.out), static_cast<const T*>(a.weightsMfma), a.bias, a.nbr,
                     static_cast<uint32_t>(pitch), a.tapMirror, a.tileMasks, a.kVol, a.inRows, a.outRows, a.relu, tiles, perBlock,
                     chip.xcdShift, a.numActOut);
  return D3D_OK;
}

}  // namespace convk
}  // namespace d3d
