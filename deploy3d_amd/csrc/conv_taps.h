// MFMA convolution for rows of at most 32 bytes (16 two-byte channels, 32 int8 channels and fewer): several taps per MFMA.
//
// An MFMA contracts 64 bytes per row.  convMfmaResident (conv_kernels.h) gives such a row an MFMA of 32 bytes to itself and
// so pays one table lookup, one gather, one set of weight reads and one scalar walk per 16 rows and tap; counted in
// instructions that, and not the memory system, is what those layers are bound by (16 -> 32 at stride 2, 1.4 million rows:
// 66 clocks per CU and (16 rows, tap), of which a gather whose rows are mostly absent needs 20).  Here the four lane
// groups of the operand layout take different taps: two of 32 bytes or four of 16 bytes per MFMA, each lane reading 16
// bytes of its own (row, tap).  Weights of all taps stay in LDS in the order the lanes read them, every wavefront walks its
// own 16-row groups without barriers.
// The table slice of a group is loaded as (tap = 4 * q + lane / 16, row = lane % 16), so taps live in slots
// (tap % 4) * Q + tap / 4: the taps that occur then come out of the sign bits of the loaded entries, a reduction over 16
// lanes and four lane reads, and one 32-bit mask is walked.  Slot 0 is the null tap (rows absent, weights zero) that fills
// up the last MFMA; the walk yields it by itself, because an empty mask has 32 leading zeros.
// Measured (convMfmaResident before), us: 5 -> 16 / 16 -> 16 fp16, 120 000 rows 8.1 (17.8) / 7.2 (12.0), 480 000 bf16 rows 21
// (48) / 19 (30); 16 -> 32 at stride 2, 349 000 rows 22 (35), 1.4 million 89 (136; of them 56 for its 256 MB at the rate of a
// large copy: table, rows in, rows out); 9 000 rows 4.7 - 6.6 (6.6 - 11.5), near a launch.  int8, 349 000 rows: 16 -> 32 at
// stride 2 25 (41), 32 -> 64 at stride 2 33 (55), 32 -> 32 with tile masks 33 (43 on convStaged).
#pragma once
#include "conv_kernels.h"

namespace d3d {
namespace convk {

// RB: bytes of a stored row, 32 or 16; 0: rowCh channels, at most eight, read as they lie.  CB: bytes of K a tap takes (a
// row padded to 16 or 32).  QC: table loads per group where known (7: a 3x3x3 kernel), 0: from kVol.
template <class T, int RB, int CB, int COUT, int QC, int WAVES>
__global__ void __launch_bounds__(64 * WAVES, COUT <= 32 ? 8 : 4)
convTaps(const T* __restrict__ in, T* __restrict__ out, const T* __restrict__ wf, const float* __restrict__ bias,
         const float* __restrict__ requantM, const int32_t* __restrict__ nbr, int64_t nbrPitch, int tapMirror, int kVol,
         int64_t inRows, int64_t outRows, int relu, int groups, int xcdShift, const int32_t* __restrict__ numActOut,
         int rowCh) {
  constexpr int ES = static_cast<int>(sizeof(T));
  constexpr int NT = COUT / 16;
  constexpr int LG = CB / 16;                          // lane groups that share a tap
  constexpr int TPM = 4 / LG;                          // taps per MFMA
  constexpr int WTAP = NT * LG * 256;                  // bytes of a tap's weights in LDS
  constexpr int MAXQ = QC ? QC : 8;                    // table loads per group: kernel volumes up to 32
  using Acc = typename Mfma<T>::Acc;
  static_assert(ES <= 2 && (CB == 16 || CB == 32) && (RB == 0 ? CB == 16 : RB == CB), "rows of at most 32 bytes");

  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int Q = QC ? QC : (kVol + 3) >> 2, slots = 4 * Q + 1;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r16 = lane & 15, kgrp = lane >> 4, part = kgrp % LG;
  int32_t* const nb = reinterpret_cast<int32_t*>(smem + slots * WTAP) + wave * slots * 16;  // [slot][16], this wavefront's

  // Weights: the packed copy is 8-byte pieces [tap][n][K group][column]; two pieces of a column make the 16 bytes a lane
  // multiplies.  Slots without a tap (the null tap, taps past the kernel volume) are zero.
  for (int e = tid; e < slots * WTAP / 16; e += 64 * WAVES) {
    const int slot = e / (WTAP / 16), tap = slot == 0 ? kVol : (slot - 1) % Q * 4 + (slot - 1) / Q;
    const int n = e / (LG * 16) % NT, p = e / 16 % LG, c = e % 16;
    u32x4 v = {0u, 0u, 0u, 0u};
    if (tap < kVol) {
      const u32x2* src = reinterpret_cast<const u32x2*>(wf) + ((tap * NT + n) * 64 + 2 * p * 16 + c);
      const u32x2 a = src[0], b = src[16];
      v = u32x4{a[0], a[1], b[0], b[1]};
    }
    reinterpret_cast<u32x4*>(smem)[e] = v;
  }
  if (lane < 16) nb[lane] = -1;
  __syncthreads();

  const int wavesPerXcd = (gridDim.x >> xcdShift) * WAVES;
  const TileOrder order(groups, static_cast<int>((liveOutRows(numActOut, outRows) + 15) / 16), xcdShift,
                        blockIdx.x & ((1 << xcdShift) - 1));
  // entry q of this lane's part of a group's table slice: tap 4 * q + kgrp
  const int64_t tapStep = (tapMirror ? -4 : 4) * nbrPitch;
  const int32_t* const tap0 = nbr + static_cast<int64_t>(tapMirror ? kVol - 1 - (kgrp < kVol ? kgrp : 0) : (kgrp < kVol ? kgrp : 0)) * nbrPitch;
  int32_t next[MAXQ];
  auto requestTable = [&](int local) __attribute__((always_inline)) {
    if (local >= order.count()) return;
    int64_t row = static_cast<int64_t>(order.tile(local)) * 16 + r16;
    if (row >= outRows) row = outRows - 1;               // its result is not stored
    const int32_t* p = tap0 + row;
#pragma unroll
    for (int q = 0; q < MAXQ; ++q) {
      if (q < Q) next[q] = 4 * q + kgrp < kVol ? p[q * tapStep] : -1;
    }
  };

  // The 16 bytes of the lane's row of neighbour `idx` (-1: zeros), as they come from memory, and as the MFMA takes them.
  // Rows of rowCh channels begin at any byte: the four aligned words around one hold it (a row of at most 14 bytes, an
  // even number of them where rows begin at even bytes), and it is shifted and cut to size where it is used, so that the
  // loads of later steps stay in flight.  An absent neighbour's offset lies past the buffer: the load returns zeros.
  const uint32_t rowBytes = RB ? RB : static_cast<uint32_t>(rowCh) * ES, rows = static_cast<uint32_t>(inRows);
  const __amdgpu_buffer_rsrc_t inBuf = makeRawBuffer(in, (static_cast<uint32_t>(inRows) * rowBytes + 3u) & ~3u);
  struct Gathered {
    u32x4 words;
    uint32_t at;
  };
  auto gather = [&](int32_t idx) __attribute__((always_inline)) -> Gathered {
    const uint32_t at = RB ? static_cast<uint32_t>(idx) * RB + part * 16u : (static_cast<uint32_t>(idx) < rows ? static_cast<uint32_t>(idx) * rowBytes : 0xC0000000u);
    return {__builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(inBuf, RB ? at : at & ~3u, 0, 0)), at};
  };
  uint32_t keep[4];                                    // bytes of the four words that a row of rowCh channels fills
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int n = static_cast<int>(rowBytes) - 4 * j;
    keep[j] = n >= 4 ? ~0u : (n <= 0 ? 0u : (1u << (8 * n)) - 1u);
  }
  auto operand = [&](const Gathered& g) __attribute__((always_inline)) -> u32x4 {
    if constexpr (RB != 0) {
      return g.words;
    } else {
      u32x4 v;
#pragma unroll
      for (int j = 0; j < 4; ++j) v[j] = __builtin_amdgcn_alignbyte(j < 3 ? g.words[j + 1] : 0u, g.words[j], g.at & 3u) & keep[j];
      return v;
    }
  };

  // bias of the channels this lane stores; the int8 layers load theirs with the scales, row group by row group
  float4v biasV[NT];
#pragma unroll
  for (int n = 0; n < NT; ++n)
    biasV[n] = ES == 2 && bias ? *reinterpret_cast<const float4v*>(bias + n * 16 + kgrp * 4) : float4v{0.f, 0.f, 0.f, 0.f};

  const int firstLocal = (blockIdx.x >> xcdShift) * WAVES + wave;
  requestTable(firstLocal);
  for (int local = firstLocal; local < order.count(); local += wavesPerXcd) {
    const int64_t row0 = static_cast<int64_t>(order.tile(local)) * 16;

    // the slice goes to LDS; a lane gathers the sign bits of its entries, the 16 lanes of a group merge theirs
    uint32_t absent = 0;                               // bit q: this lane group's tap 4 * q + kgrp has no row
#pragma unroll
    for (int q = MAXQ - 1; q >= 0; --q) {
      if (q < Q) {
        nb[(1 + kgrp * Q + q) * 16 + r16] = next[q];
        absent = (absent << 1) | (static_cast<uint32_t>(next[q]) >> 31);
      }
    }
#define D3D_ROW_AND(CTRL) absent &= static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(absent), CTRL, 0xF, 0xF, false))
    D3D_ROW_AND(0x128);                                // row_ror:8, 4, 2, 1
    D3D_ROW_AND(0x124);
    D3D_ROW_AND(0x122);
    D3D_ROW_AND(0x121);
#undef D3D_ROW_AND
    const uint32_t have = ~absent & ((1u << Q) - 1u);
    uint32_t active = 0;                               // bit s: slot 1 + s occurs in the group
#pragma unroll
    for (int g = 0; g < 4; ++g) active |= static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(have), 16 * g)) << (g * Q);
    auto nextSlot = [&]() __attribute__((always_inline)) -> int {   // highest first; 0 once the list is exhausted
      active = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(active)));  // stays scalar
      const uint32_t zeros = active ? static_cast<uint32_t>(__builtin_clz(active)) : 32u;
      active &= ~(0x80000000u >> (zeros & 31u));
      return 32 - static_cast<int>(zeros);
    };
    // the slot this lane multiplies in the next MFMA
    auto laneSlot = [&]() __attribute__((always_inline)) -> int {
      if constexpr (TPM == 2) {
        const int a = nextSlot(), b = nextSlot();
        return kgrp >= 2 ? b : a;
      } else {
        const int a = nextSlot(), b = nextSlot(), c = nextSlot(), d = nextSlot();
        const int ab = kgrp & 1 ? b : a, cd = kgrp & 1 ? d : c;
        return kgrp & 2 ? cd : ab;
      }
    };

    Acc acc[NT];
#pragma unroll
    for (int n = 0; n < NT; ++n) acc[n] = Acc{0, 0, 0, 0};
    const unsigned char* const wLane = smem + part * 256 + r16 * 16;
    auto multiply = [&](int slot, const Gathered& g) __attribute__((always_inline)) {
      const unsigned char* w = wLane + slot * WTAP;
      const u32x4 rows = operand(g);
#pragma unroll
      for (int n = 0; n < NT; ++n)
        acc[n] = Mfma<T>::k32(*reinterpret_cast<const u32x4*>(w + n * LG * 256), rows, acc[n]);
    };

    int steps = (__builtin_popcount(active) + TPM - 1) / TPM;
    int sA = laneSlot(), sB = laneSlot(), sC;
    Gathered bufA = gather(nb[sA * 16 + r16]), bufB = gather(nb[sB * 16 + r16]), bufC;
    requestTable(local + wavesPerXcd);
    // three steps per iteration, no branch between them (see convMfma)
    for (; steps > 0; steps -= 3) {
      sC = laneSlot();
      bufC = gather(nb[sC * 16 + r16]);
      __builtin_amdgcn_sched_barrier(0);
      multiply(sA, bufA);
      __builtin_amdgcn_sched_barrier(0);
      sA = laneSlot();
      bufA = gather(nb[sA * 16 + r16]);
      __builtin_amdgcn_sched_barrier(0);
      multiply(sB, bufB);
      __builtin_amdgcn_sched_barrier(0);
      sB = laneSlot();
      bufB = gather(nb[sB * 16 + r16]);
      __builtin_amdgcn_sched_barrier(0);
      multiply(sC, bufC);
      __builtin_amdgcn_sched_barrier(0);
    }

    const int64_t row = row0 + r16;
    if (row < outRows) {
#pragma unroll
      for (int n = 0; n < NT; ++n) {
        const int col = n * 16 + kgrp * 4;
        if constexpr (ES == 1) {
          // int8: t = float(acc) * m[c]; t += bq[c]; round to nearest even; clamp (lo = 0 with the fused ReLU)
          const float4v mq = *reinterpret_cast<const float4v*>(requantM + col), bq = *reinterpret_cast<const float4v*>(bias + col);
          uint32_t packed = 0;
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            float t = static_cast<float>(acc[n][j]) * mq[j];
            t = t + bq[j];
            float v = __builtin_rintf(t);
            v = __builtin_fminf(127.f, __builtin_fmaxf(relu ? 0.f : -128.f, v));
            packed |= (static_cast<uint32_t>(static_cast<int>(v)) & 0xFFu) << (8 * j);
          }
          *reinterpret_cast<uint32_t*>(out + static_cast<size_t>(row) * COUT + col) = packed;
        } else {
          T packed[4];
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            float v = acc[n][j] + biasV[n][j];
            if (relu) v = v > 0.f ? v : 0.f;
            packed[j] = static_cast<T>(v);
          }
          *reinterpret_cast<u32x2*>(out + static_cast<size_t>(row) * COUT + col) = __builtin_bit_cast(u32x2, packed);
        }
      }
    }
  }
}

constexpr int kTapsWaves = 16;
inline size_t tapsLds(int kVol, int tapBytes, int cout) {
  return static_cast<size_t>((kVol + 3) / 4 * 4 + 1) * (tapBytes * cout + kTapsWaves * 64);
}

inline bool tapsFit(int kVol, int tapBytes, int cout) { return kVol <= 32 && tapsLds(kVol, tapBytes, cout) <= kLdsLimit; }

// 32-bit row offsets, with room above them for the one of an absent neighbour
inline bool tapsReach(int64_t rows, uint64_t rowBytes) { return static_cast<uint64_t>(rows) * rowBytes < 0xBFFF0000ull; }

template <class T, int RB, int CB, int COUT, int QC>
int32_t launchTapsCfg(const ConvArgs& a, hipStream_t stream) {
  constexpr int WAVES = kTapsWaves;
  const size_t lds = tapsLds(a.kVol, CB, COUT);
  if (!tapsFit(a.kVol, CB, COUT) || !tapsReach(a.inRows, RB ? RB : a.rowChannels * sizeof(T))) return D3D_ERR_UNSUPPORTED;
  static std::atomic<size_t> granted{64 * 1024};
  const int32_t rc = grantLds(&convTaps<T, RB, CB, COUT, QC, WAVES>, lds, &granted);
  if (rc != D3D_OK) return rc;
  const int groups = static_cast<int>((a.outRows + 15) / 16);
  const ChipLayout chip = chipLayout();
  const int nXcd = 1 << chip.xcdShift;
  int perCu = static_cast<int>(kLdsLimit / (lds + 1024));
  perCu = perCu < 1 ? 1 : (perCu > 2 ? 2 : perCu);   // 16 wavefronts each
  int blocks = chip.cus / nXcd * nXcd * perCu;
  const int needed = (groups + WAVES - 1) / WAVES;
  if (blocks > needed) blocks = (needed + nXcd - 1) / nXcd * nXcd;
  hipLaunchKernelGGL((convTaps<T, RB, CB, COUT, QC, WAVES>), dim3(static_cast<unsigned>(blocks)), dim3(64 * WAVES), lds, stream,
                     static_cast<const T*>(a.in), static_cast<T*>(a.out), static_cast<const T*>(a.weightsMfma), a.bias,
                     a.requantM, a.nbr, a.nbrPitch > 0 ? a.nbrPitch : a.outRows, a.tapMirror, a.kVol, a.inRows, a.outRows,
                     a.relu, groups, chip.xcdShift, a.numActOut, a.rowChannels);
  return D3D_OK;
}

template <class T, int RB, int CB, int COUT>
int32_t launchTaps(const ConvArgs& a, hipStream_t stream) {
  if (a.kVol > 24 && a.kVol <= 28) return launchTapsCfg<T, RB, CB, COUT, 7>(a, stream);
  return launchTapsCfg<T, RB, CB, COUT, 0>(a, stream);
}

}  // namespace convk
}  // namespace d3d
