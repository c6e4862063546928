// Software-pipelined MFMA convolution for gfx950 (fp16 / bf16 storage with fp32 accumulation; int8 storage with
// int32 accumulation and a requantizing store, for rows of 64 or 128 bytes; fp32).
//
// Same mathematics and data layouts as convStaged (conv_kernels.h): output-stationary tiles, rows of a tap
// gathered through the neighbour table into an XOR-swizzled LDS stage, weights in fragment-major order streamed
// through LDS, one plain store per output element.  What differs is the schedule.  convStaged runs 8 wavefronts
// that a barrier re-aligns every tap, each with its phases back to back (weight fragments from LDS, MFMAs,
// gather issue, row fragments from LDS), so the LDS pipe, the vector-memory path and the matrix pipe take turns,
// and every tile pays for a prologue of two dependent memory round trips.  Here
//  * a wavefront multiplies its 16*MT rows one 16-row group after the other and keeps two register sets of
//    fragments: while group m multiplies, the row fragments of group m+1 and one weight fragment of the NEXT step
//    are read from LDS, the stage rows of group m (already in registers) are refilled with the rows of the step
//    after next, and the index and weight loads of later steps are issued - each piece placed behind an MFMA in
//    program order, so all of it runs in the shadow of the matrix pipe;
//  * workgroups are persistent and the pipeline runs ACROSS tiles: a workgroup's tiles form one stream of steps
//    (tile, tap, channel part); when the multiplying end of the pipeline finishes a tile it stores the tile's rows
//    and clears the accumulators, while the loading end is already several steps into the next tile.  Only the
//    first tile of a workgroup pays for a prologue;
//  * a step exists only for taps that some row of the workgroup's tile has (tile masks written with the table).
//
// Gathers and index loads are buffer loads: an absent neighbour (-1) or a row past the input produces an
// out-of-range offset, for which the hardware delivers zeros - no zero row, no select, one VALU per gather.
#pragma once
#include <cstring>
#include <type_traits>

#include "conv_kernels.h"
#include "deal.h"

namespace d3d {
namespace convk {

typedef __attribute__((address_space(3))) void* LdsVoidPtr;

// Workgroups that take all 128 output channels of their rows, in wavefronts of 32 rows: the tile (256, 192 or 128 rows) that
// loads the busiest of `cus` CUs least with `rows` rows (rounds of tiles x rows per tile); see launchPipeShape.
__device__ inline int pipeTileRows(int64_t rows, int cus) {
  auto load = [&](int tile) { return static_cast<int>((rows + static_cast<int64_t>(tile) * cus - 1) / (static_cast<int64_t>(tile) * cus)) * tile; };
  const int l8 = load(256), l6 = load(192), l4 = load(128);
  const int best = l6 < l8 ? 192 : 256;
  return l4 < (l6 < l8 ? l6 : l8) ? 128 : best;
}

// The tiles one of `per` workgroups of an XCD takes, in order.  A tile's time goes by the taps its rows have (27, or 18 and 9
// in the outer levels of a scene), and a layer ends with its busiest workgroup.  Where workgroups take several tiles and masks
// say what those hold, the tiles of an XCD are ranked by their taps, most first, and dealt back and forth: one with a heavy
// tile gets a light one with it.  XCDs take runs of up to CHUNK tiles in turn instead of a contiguous eighth each, which could
// be all heavy: levels of a scene are contiguous.  (Runs are short enough for sixteen turns: with 16-tile runs 195 tiles are 32 for
// five XCDs and 16 for three.)  Each wavefront ranks for itself, 64 tiles to a register, and keeps its
// workgroup's list in the lanes of one register.
// Otherwise (no masks, at most ROUNDS tiles each or more than a list holds) XCD x takes the x-th contiguous part (TileOrder).
// fp32 layers, bound by the matrix pipe, are dealt from the second tile on: steps of the busiest workgroup / of the average
// one 153 / 110 contiguous and 120 / 110 dealt for 64 -> 64 with 260 000 rows, 407 -> 344 us; 118 000 rows 208 -> 174.  Two-byte
// layers of 64 input channels and more gain from the fifth tile on (64 -> 64, 1.04 million rows of a network's third level, 216 / 174 ->
// 180 / 174 steps: 228 -> 210 us; 64 -> 128 451 -> 430, 128 -> 64 431 -> 395, 128 -> 32 354 -> 327) and not before: with two tiles each
// (260 000 rows, 54 / 44 -> 45 / 44) the part runs at a lower clock when no CU is idle, the XCDs read 20 % more lines from each other's
// parts, and it was 58.7 against 59.2 us alone and 25 us of 630 lost in a pass whose rulebooks had run on the CUs that finished early.
// Those lines are the price everywhere: rows in a scan's own order, whose tiles all hold much the same taps, lose by it (64 -> 64, 1.08
// million rows 227 -> 243 us), but layers of 64 channels have a level's rows.  int8 and 32 two-byte input channels, three workgroups to
// a CU, only pay: int8 64 -> 128, 520 000 rows 122 us contiguous, 130 dealt, 1.04 million 267 and 271, 64 -> 64 840 000 rows of scans 86
// and 96, a level's 1.04 million 115 to 118 either way; 32 -> 64 in bf16, 1.4 million rows 214 and 216, 840 000 of scans 94 and 100.
constexpr int kDealRounds = 4;
template <int PER, int CHUNK, int ROUNDS>                // ROUNDS = 0: never dealt
struct TileDeal {
  static constexpr int SLOTS = 4;                        // registers of tiles ranked together
  TileOrder order;
  int first, per, mine, list;                            // list: lane p holds the tile of turn p, `mine` of them
  bool dealt;
  __device__ __forceinline__ TileDeal(int tiles, int live, int xcdShift, int xcd, int first_, int per_,
                                      const unsigned long long* __restrict__ tileMasks, int kVol, unsigned long long allTaps, int lane)
      : order(tiles, live, xcdShift, xcd), first(first_), per(per_), mine(0), list(0), dealt(false) {
    if constexpr (ROUNDS > 0) deal(xcdShift, xcd, tileMasks, kVol, allTaps, lane);
  }
  __device__ __forceinline__ void deal(int xcdShift, int xcd, const unsigned long long* __restrict__ tileMasks, int kVol,
                                       unsigned long long allTaps, int lane) {
    const int live = order.liveTiles, wgs = per << xcdShift;
    if (!tileMasks || live <= ROUNDS * wgs || live > 32 * wgs || per > 192) return;
    dealt = true;
    int cs = 0;                                          // log2 of a run's tiles
    while ((2 << cs) <= CHUNK && (2 << cs) <= live >> (xcdShift + 4)) ++cs;
    const int chunks = ((live - 1) >> cs) + 1;
    int lx = ((chunks - xcd + order.nXcd - 1) >> xcdShift) << cs;     // chunks xcd, xcd + nXcd, ...; the last one may be short
    if (((chunks - 1) & (order.nXcd - 1)) == xcd) lx -= (chunks << cs) - live;
    if (lx < 0) lx = 0;
    for (int from = 0; from < lx; from += 64 * SLOTS) {
      int taps[SLOTS], at[SLOTS], rank[SLOTS];
#pragma unroll
      for (int s = 0; s < SLOTS; ++s) {
        const int local = from + s * 64 + lane;
        at[s] = ((((local >> cs) << xcdShift) + xcd) << cs) + (local & ((1 << cs) - 1));
        taps[s] = -1;
        rank[s] = 0;
        if (local < lx) {
          unsigned long long m = 0;
#pragma unroll
          for (int e = 0; e < PER; ++e) m |= tileMasks[static_cast<int64_t>(at[s]) * PER + e];
          taps[s] = __builtin_popcountll(m & allTaps);
        }
      }
      int base = 0;
      for (int c = kVol; c >= 0; --c) {
#pragma unroll
        for (int s = 0; s < SLOTS; ++s) {
          const unsigned long long b = __ballot(taps[s] == c);
          if (b) {
            const int before = __builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(b >> 32), __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(b), 0u));
            if (taps[s] == c) rank[s] = base + before;
            base += __builtin_popcountll(b);
          }
        }
      }
#pragma unroll
      for (int s = 0; s < SLOTS; ++s) {
        const DealtTile to = dealTile(from, rank[s], per);
        unsigned long long b = __ballot(taps[s] >= 0 && to.workgroup == first);
        for (; b; b &= b - 1) {
          const int l = __builtin_ctzll(b);
          const int turn = __builtin_amdgcn_readlane(to.turn, l), t = __builtin_amdgcn_readlane(at[s], l);
          if (lane == turn) list = t;
          ++mine;
        }
      }
    }
    mine = __builtin_amdgcn_readfirstlane(mine);
  }
  // tiles of this workgroup: the live ones, then its share of those past the live rows
  __device__ __forceinline__ int count() const {
    if constexpr (ROUNDS == 0) return first < order.count() ? (order.count() - 1 - first) / per + 1 : 0;
    const int n = dealt ? order.dx : order.count();
    return mine + (first < n ? (n - 1 - first) / per + 1 : 0);
  }
  __device__ __forceinline__ bool live(int pos) const { return ROUNDS > 0 && dealt ? pos < mine : order.live(first + pos * per); }
  __device__ __forceinline__ int tile(int pos) const {
    if (ROUNDS == 0 || !dealt) return order.tile(first + pos * per);
    if (pos < mine) return __builtin_amdgcn_readlane(list, pos);
    return order.liveTiles + (first + (pos - mine) * per) * order.nXcd + order.xcd;
  }
};

// tileMasks: one 64-bit tap mask per 64 output rows, padded with zero entries to a multiple of 8 entries past
// ceil(outRows / 64) (a workgroup reads the masks of a whole tile at once); null = every tap of every tile.
//
// SPLIT = 2: a tile is the work of two groups of WAVES wavefronts, each with half of the steps and LDS of its own (channel
// halves of every tap where a tap takes two steps, else half of the tile's taps); the second group's sums pass through its stage
// to the first, which adds and stores them.
template <class T, int CIN, int COUT, int MT, int WAVES, int CO = COUT, bool DEAL = false, int SPLIT = 1>
__device__ __forceinline__ void
pipeTiles(unsigned char* smem, const T* __restrict__ in, T* __restrict__ out, const T* __restrict__ wf,
          const float* __restrict__ bias, const float* __restrict__ requantM, const int32_t* __restrict__ nbr, int64_t nbrPitch,
          int tapMirror, const unsigned long long* __restrict__ tileMasks, int kVol, int64_t inRows, int64_t outRows, int relu,
          int xcdShift, const int32_t* __restrict__ numActOut, int blocks, const int32_t* __restrict__ rowOrder = nullptr) {
  constexpr int THREADS = 64 * WAVES;
  constexpr int ES = static_cast<int>(sizeof(T));
  constexpr int CS = CIN * ES > 128 ? 128 / ES : CIN;          // input channels per step (at most 128 bytes of a row); a tap takes KS steps
  constexpr int KS = CIN / CS;
  constexpr int CH = CS * ES / 16;                             // 16-byte chunks of a row staged per step
  constexpr int RPI = 64 / CH;                                 // rows one gather instruction covers
  constexpr int WM = 16 * MT, TM = WAVES * WM;
  constexpr int GL = WM / RPI;                                 // gather instructions per step
  constexpr int GPM = 16 / RPI;                                // gathers that cover the 16 rows of one row group
  constexpr int NT = CO / 16;
  constexpr int COLS = COUT / CO;                              // workgroups that share a tile, CO output channels each
  constexpr int KK = CS * ES / 64;                             // MFMAs along K per step: 64 bytes of a row each
  constexpr int NQ = KK * NT;                                  // MFMAs per row group and step
  constexpr int WCH = CS * CO * ES / 16;                       // 16-byte chunks of one step's weights
  constexpr int WL = (WCH + THREADS - 1) / THREADS;            // weight loads per wavefront and step
  constexpr int NWB = 3;                                       // weight buffers
  constexpr int NI = 4;                                        // index ring depth (steps)
  constexpr int IL = (WM + 63) / 64;                           // index loads per step
  constexpr int SLOTS = WM * CH;                               // 16-byte slots of one stage
  constexpr int PER = TM / 64;                                 // tile masks per workgroup tile
  constexpr int ROWSHIFT = CIN * ES == 64 ? 6 : (CIN * ES == 128 ? 7 : (CIN * ES == 256 ? 8 : 9));
  static_assert((ES == 4 || ES == 2 || ES == 1) && (CS * ES == 64 || CS * ES == 128) && CIN % CS == 0 && WM % RPI == 0 && TM % 64 == 0, "shape");
  static_assert((1 << ROWSHIFT) == CIN * ES && WCH % 64 == 0 && MT >= 2 && MT * NT * 4 <= 128, "shape");
  static_assert(WM < 64 || WM % 64 == 0, "an index load covers 64 rows: a wavefront tile is below 64 rows or whole multiples");
  using F = u32x4;
  using Acc = typename Mfma<T>::Acc;

  constexpr int SPT = SPLIT > 1 && KS > 1 ? KS / SPLIT : KS;   // steps of a tap in one group
  static_assert(SPLIT == 1 || (SPLIT == 2 && !DEAL && KS <= 2 && MT * NT * 1024 <= 2 * SLOTS * 16), "two groups, whose sums fit a stage");

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6) % WAVES;
  const int group = SPLIT > 1 ? __builtin_amdgcn_readfirstlane(tid >> 6) / WAVES : 0;
  const int r16 = lane & 15, kgrp = lane >> 4;
  if constexpr (SPLIT > 1) smem += group * (NWB * WCH * 16 + WAVES * (2 * SLOTS * 16 + NI * WM * 4));
  u32x4* wLds = reinterpret_cast<u32x4*>(smem);                                      // [NWB][WCH]
  u32x4* stage = reinterpret_cast<u32x4*>(smem + static_cast<size_t>(NWB) * WCH * 16) + wave * 2 * SLOTS;  // [2][SLOTS]
  // ring of NI steps' neighbour indices, per wavefront, stored so that the GL indices one lane needs for its
  // gathers are consecutive: position (lane / CH) * GL + j holds the index of tile row j * RPI + lane / CH
  int32_t* idxLds = reinterpret_cast<int32_t*>(smem + static_cast<size_t>(NWB) * WCH * 16 +
                                               static_cast<size_t>(WAVES) * 2 * SLOTS * 16) + wave * NI * WM;

  // the 16-byte chunk of a row this lane gathers: logical chunk (lane % CH) of stage row (j * RPI + lane / CH)
  // lands in physical chunk lane % CH, so the lane fetches the chunk that the swizzle maps there (the swizzle of
  // a stage row does not depend on j)
  const uint32_t chunkOff = static_cast<uint32_t>(((lane % CH) ^ stageSwizzle<CH>(lane / CH)) * 16);
  const __amdgpu_buffer_rsrc_t inBuf = makeRawBuffer(in, static_cast<uint32_t>(inRows * (CIN * ES)));
  const __amdgpu_buffer_rsrc_t nbrBuf = makeRawBuffer(nbr, static_cast<uint32_t>(kVol * nbrPitch * 4));
  // Row of the tile (counted from the workgroup's first row) whose index sits at ring position i * 64 + lane:
  // position p belongs to the wavefront's row (p % GL) * RPI + p / GL.
  uint32_t idxRow[IL];
#pragma unroll
  for (int i = 0; i < IL; ++i) {
    const int p = i * 64 + lane;
    idxRow[i] = static_cast<uint32_t>(wave * WM + (p % GL) * RPI + p / GL);
  }

  // ---- this workgroup's tiles (TileDeal) ----
  const int part = (blockIdx.x >> xcdShift) % COLS;      // which CO of the output channels
  const unsigned long long allTaps = kVol >= 64 ? ~0ull : ((1ull << kVol) - 1ull);
  const TileDeal<PER, (TM < 2048 ? 2048 / TM : 1), DEAL ? (ES == 4 ? 1 : kDealRounds) : 0> deal(
      static_cast<int>((outRows + TM - 1) / TM), static_cast<int>((liveOutRows(numActOut, outRows) + TM - 1) / TM), xcdShift,
      blockIdx.x & ((1 << xcdShift) - 1), (blockIdx.x >> xcdShift) / COLS, (blocks >> xcdShift) / COLS, tileMasks, kVol, allTaps, lane);
  const int nMine = deal.count();
  if (nMine <= 0) return;                                // workgroup-uniform
  auto tileAt = [&](int pos) __attribute__((always_inline)) { return deal.tile(pos); };
  // taps of the workgroup's pos-th tile; a tile without any tap still takes one step (tap 0: all rows absent)
  auto maskAt = [&](int pos) __attribute__((always_inline)) -> unsigned long long {
    if (pos >= nMine) return 0ull;
    if (!deal.live(pos)) return 1ull;                    // no live row: one step of absent neighbours
    unsigned long long m = allTaps;
    if (tileMasks) {
      const unsigned long long* p = tileMasks + static_cast<int64_t>(tileAt(pos)) * PER;
      m = 0;
#pragma unroll
      for (int e = 0; e < PER; ++e) m |= p[e];
      m &= allTaps;
    }
    return m ? m : 1ull;
  };

  // The workgroup's steps (tile, tap, part) in order.  One walk serves all consumers: the index loads run four steps
  // ahead of the multiplication, the weight loads three, the gathers two, so a step's id is made once, by the index
  // load, and handed down a chain of scalars (a walk per consumer took a third of a 32-channel step's instructions).
  // Past the last step the walk stays on it: the loads issued for steps that do not exist repeat valid addresses and
  // nothing in the loop has to branch on "is there such a step".
  constexpr uint32_t kLastOfTile = 1u << 31;
  // (two groups: tile by tile, each with a pipeline of its own)
  for (int firstPos = 0; firstPos < (SPLIT > 1 ? nMine : 1); ++firstPos) {
  const int endPos = SPLIT > 1 ? firstPos + 1 : nMine;
  int walkPos = firstPos;                            // ordinal of the walk's tile among this workgroup's
  unsigned long long walkRem = maskAt(firstPos), walkTaps = SPLIT > 1 ? 0ull : maskAt(1);  // taps of it still to walk; taps of the next tile
  int mySteps = 0, mostSteps = 0;                    // steps of this group / of the group that has more
  if constexpr (SPLIT > 1) {
    const int taps = __builtin_popcountll(walkRem);
    mySteps = mostSteps = taps * SPT;
    if constexpr (KS == 1) {                         // the lower half of the taps, rounded up, is the first group's
      unsigned long long upper = walkRem;
      for (int i = 0; i < (taps + 1) / 2; ++i) upper &= upper - 1;
      walkRem = group ? upper : walkRem ^ upper;
      mostSteps = (taps + 1) / 2;
      mySteps = group ? taps / 2 : mostSteps;
    }
  }
  int walkTap = 0, walkPart = 0;
  // moves to the next step; returns its id (tap * KS + part), flagged when it ends its tile.  *newTile = it opens one.
  auto walkNext = [&](bool* newTile) __attribute__((always_inline)) -> uint32_t {
    *newTile = false;
    if (walkPart == 0) {
      if (walkRem == 0 && walkPos + 1 < endPos) {
        ++walkPos;
        walkRem = walkTaps;
        walkTaps = maskAt(walkPos + 1);
        *newTile = true;
      }
      if (walkRem) {
        walkTap = __builtin_ctzll(walkRem);
        walkRem &= walkRem - 1;
      }
    }
    const uint32_t s = static_cast<uint32_t>(walkTap * KS + walkPart + (SPT < KS ? group * SPT : 0));
    walkPart = walkPart + 1 == SPT ? 0 : walkPart + 1;
    return s | (walkRem == 0 && walkPart == 0 ? kLastOfTile : 0u);
  };
  uint32_t ids[5];                                   // steps a .. a+4
  int mulPos = 0;                                    // ordinal of the tile that multiplies

  F rowBuf[2][KK];                                   // row fragments of the group that multiplies / of the next
  int32_t ixBuf[2][GPM];                             // neighbour indices for the gathers of this group / the next
  F wtsA[KK][NT], wtsB[KK][NT];                      // weight fragments of this step / of the next
  Acc acc[MT][NT];
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int n = 0; n < NT; ++n) acc[m][n] = Acc{0, 0, 0, 0};

  // indices of the index walk's next step -> ring slot `seq % NI` (asynchronous, straight into LDS); rows past
  // the table read as 0 and are never stored
  uint32_t idxOff[IL];
  auto loadIndex = [&](int seq) __attribute__((always_inline)) -> uint32_t {
    bool newTile;
    const uint32_t id = walkNext(&newTile);
    const int tap = walkTap;
    if (newTile || seq == 0) {
      const uint32_t rowBase = static_cast<uint32_t>(tileAt(walkPos)) * TM;
#pragma unroll
      for (int i = 0; i < IL; ++i) idxOff[i] = (rowBase + idxRow[i]) * 4u;
    }
    const uint32_t base = static_cast<uint32_t>((tapMirror ? kVol - 1 - tap : tap) * nbrPitch * 4);
#pragma unroll
    for (int i = 0; i < IL; ++i) {
      if (WM >= 64 || lane < WM)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(nbrBuf, (LdsVoidPtr)(idxLds + (seq & (NI - 1)) * WM + i * 64), 4,
                                                 base + idxOff[i], 0, 0, 0);
    }
    return id;
  };
  // the GPM indices of row group m of ring slot `seq % NI`, for this lane's gathers
  auto readIndex = [&](int seq, int m, int32_t (&dst)[GPM]) __attribute__((always_inline)) {
    const int32_t* p = idxLds + (seq & (NI - 1)) * WM + (lane / CH) * GL + m * GPM;
    if constexpr (GPM == 2) {
      const u32x2 v = *reinterpret_cast<const u32x2*>(p);
      dst[0] = static_cast<int32_t>(v[0]);
      dst[1] = static_cast<int32_t>(v[1]);
    } else {
      dst[0] = *p;
    }
  };
  auto gatherOne = [&](int j, int32_t idx, uint32_t partOff, int slot) __attribute__((always_inline)) {
    const uint32_t off = (static_cast<uint32_t>(idx) << ROWSHIFT) + partOff;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(inBuf, (LdsVoidPtr)(stage + slot * SLOTS + j * 64), 16, off, 0, 0, 0);
  };
  // Buffer loads, not global ones: the compiler takes a global load into LDS for a flat access that may be pending in either
  // memory, and from then on waits for ALL outstanding LDS reads where it needs the oldest - the reads meant to run in the
  // shadow of a group's MFMAs were waited for in front of them (fp16 128 -> 128, 24 500 rows 28 -> 25.5 us, 190 000 rows
  // 135 -> 125; 64 -> 64, 262 000 rows 59.5 -> 57.5; fp32 64 -> 64, 144 000 rows 253 -> 238).
  const __amdgpu_buffer_rsrc_t wBuf = makeRawBuffer(wf, static_cast<uint32_t>(kVol * KS) * (WCH * COLS * 16u));
  auto weightLoad = [&](int q, int s, int buf) __attribute__((always_inline)) {
    const int base = (q * THREADS + wave * 64) % WCH;  // wavefronts past the slice repeat a part of it: same bytes
    // fragments lie in the order (K, channel tile): the workgroup's NT of the COLS * NT tiles of every K
    const int from = COLS == 1 ? base : (base / (NT * 64) * COLS + part) * (NT * 64) + base % (NT * 64);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(wBuf, (LdsVoidPtr)(wLds + buf * WCH + base), 16, lane * 16,
                                             (s * (WCH * COLS) + from) * 16, 0, 0);
  };
  auto readRowGroup = [&](F (&dst)[KK], int m, int slot) __attribute__((always_inline)) {
    const int n = m * 16 + r16;
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) dst[kk] = stage[slot * SLOTS + n * CH + ((kk * 4 + kgrp) ^ stageSwizzle<CH>(n))];
  };
  auto readWeight = [&](F (&dst)[KK][NT], int e, int buf) __attribute__((always_inline)) {
    dst[e / NT][e % NT] = wLds[buf * WCH + e * 64 + lane];
  };
  // Stores the finished tile (bias, ReLU, one rounding) and clears the accumulators for the next one.  After the
  // MFMAs a lane holds, per channel tile n, 4 consecutive channels (8 bytes) of one row; two 16-lane row swaps
  // per pair of channel tiles hand every lane 8 consecutive channels instead, so a store instruction writes
  // 16 bytes per lane and 64 contiguous bytes per row.
  // (fp32: 4 consecutive channels are those 16 bytes already.)
  static_assert(NT % 2 == 0 || ES == 4, "channel tiles are stored in pairs");
  // output row of the table's row (below outRows)
  auto outRow = [&](int64_t row) __attribute__((always_inline)) -> size_t {
    if constexpr (DEAL)
      if (rowOrder) return static_cast<size_t>(rowOrder[row]);
    return static_cast<size_t>(row);
  };
  auto storeTile = [&](int pos) __attribute__((always_inline)) {
    const int64_t row0 = static_cast<int64_t>(tileAt(pos)) * TM + wave * WM;
    if constexpr (ES == 4) {
#pragma unroll
      for (int n = 0; n < NT; ++n) {
        const int col = part * CO + n * 16 + kgrp * 4;
        const float4v b = bias ? *reinterpret_cast<const float4v*>(bias + col) : float4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int m = 0; m < MT; ++m) {
          float4v v;
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            v[j] = acc[m][n][j] + b[j];
            if (relu) v[j] = v[j] > 0.f ? v[j] : 0.f;
          }
          acc[m][n] = Acc{0, 0, 0, 0};
          const int64_t row = row0 + m * 16 + r16;
          if (row < outRows) *reinterpret_cast<float4v*>(out + outRow(row) * COUT + col) = v;
        }
      }
    } else {
#pragma unroll
    for (int n = 0; n < NT; n += 2) {
      const int col0 = part * CO + n * 16 + kgrp * 4, col1 = col0 + 16;
      const float4v b0 = bias ? *reinterpret_cast<const float4v*>(bias + col0) : float4v{0.f, 0.f, 0.f, 0.f};
      const float4v b1 = bias ? *reinterpret_cast<const float4v*>(bias + col1) : float4v{0.f, 0.f, 0.f, 0.f};
      // channels this lane stores after the swaps: tile n for even 16-lane rows, tile n+1 for odd ones; the
      // first or second half of the tile's 16 channels by lane row / 2
      const int outCol = part * CO + (n + (kgrp & 1)) * 16 + (kgrp >> 1) * 8;
      if constexpr (ES == 1) {
        // int8: q = clamp(rint(float(acc) * m[c] + bq[c])), lower bound 0 with the fused ReLU; a lane's 4 channels
        // are one dword, and one swap hands every lane 8 consecutive channels.  One channel tile at a time, so that
        // only one set of scales is live beside the accumulators.
        const float lo = relu ? 0.f : -128.f;
        uint32_t packed[2][MT];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int col = h ? col1 : col0;
          const float4v mq = *reinterpret_cast<const float4v*>(requantM + col);
          const float4v bq = h ? b1 : b0;
#pragma unroll
          for (int m = 0; m < MT; ++m) {
            uint32_t w = 0;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
              float t = static_cast<float>(acc[m][n + h][j]) * mq[j];
              t = t + bq[j];
              const float q = __builtin_fminf(127.f, __builtin_fmaxf(lo, __builtin_rintf(t)));
              w |= (static_cast<uint32_t>(static_cast<int>(q)) & 0xFFu) << (8 * j);
            }
            packed[h][m] = w;
            acc[m][n + h] = Acc{0, 0, 0, 0};
          }
          __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int m = 0; m < MT; ++m) {
          const auto sw = __builtin_amdgcn_permlane16_swap(packed[0][m], packed[1][m], false, false);
          const u32x2 line = {sw[0], sw[1]};
          const int64_t row = row0 + m * 16 + r16;
          if (row < outRows) *reinterpret_cast<u32x2*>(out + outRow(row) * COUT + outCol) = line;
        }
        __builtin_amdgcn_sched_barrier(0);
      } else {
#pragma unroll
      for (int m = 0; m < MT; ++m) {
        float v0[4], v1[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          v0[j] = acc[m][n][j] + b0[j];
          v1[j] = acc[m][n + 1][j] + b1[j];
          if (relu) {
            v0[j] = v0[j] > 0.f ? v0[j] : 0.f;
            v1[j] = v1[j] > 0.f ? v1[j] : 0.f;
          }
        }
        acc[m][n] = Acc{0, 0, 0, 0};
        acc[m][n + 1] = Acc{0, 0, 0, 0};
        T p0[4] = {static_cast<T>(v0[0]), static_cast<T>(v0[1]), static_cast<T>(v0[2]), static_cast<T>(v0[3])};
        T p1[4] = {static_cast<T>(v1[0]), static_cast<T>(v1[1]), static_cast<T>(v1[2]), static_cast<T>(v1[3])};
        const u32x2 a = __builtin_bit_cast(u32x2, p0), c = __builtin_bit_cast(u32x2, p1);
        // swap the odd 16-lane rows of `a` with the even ones of `c`: lane rows then hold
        //   (tile n, ch 0-3 | 4-7), (tile n+1, ch 0-3 | 4-7), (tile n, ch 8-11 | 12-15), (tile n+1, ch 8-11 | 12-15)
        const auto s0 = __builtin_amdgcn_permlane16_swap(a[0], c[0], false, false);
        const auto s1 = __builtin_amdgcn_permlane16_swap(a[1], c[1], false, false);
        const u32x4 line = {s0[0], s1[0], s0[1], s1[1]};
        const int64_t row = row0 + m * 16 + r16;
        if (row < outRows) *reinterpret_cast<u32x4*>(out + outRow(row) * COUT + outCol) = line;
      }
      }
    }
    }
  };

  // ---- prologue: indices of steps 0..3, weights of steps 0..2, rows of steps 0 and 1 in flight ----
#pragma unroll
  for (int t = 0; t < 4; ++t) ids[t] = loadIndex(t);
#pragma unroll
  for (int t = 0; t < 3; ++t) {
#pragma unroll
    for (int q = 0; q < WL; ++q) weightLoad(q, static_cast<int>(ids[t] & ~kLastOfTile), t);
  }
  waitVmcnt<0>();
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    const int s0 = static_cast<int>(ids[t] & ~kLastOfTile);
    const uint32_t p0 = chunkOff + static_cast<uint32_t>((s0 % KS) * CS * ES);
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      int32_t ix[GPM];
      readIndex(t, m, ix);
#pragma unroll
      for (int g = 0; g < GPM; ++g) gatherOne(m * GPM + g, ix[g], p0, t);
    }
  }
  waitVmcnt<0>();
  __syncthreads();                                  // the weight slices are whole
  readRowGroup(rowBuf[0], 0, 0);
  readIndex(2, 0, ixBuf[0]);
#pragma unroll
  for (int e = 0; e < NQ; ++e) readWeight(wtsA, e, 0);
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();                     // buffer 0 has been read by everyone: step 0 refills it

  // One step = one (tile, tap, channel part).  Row groups of 16 rows multiply one after the other; while group m
  // multiplies, the fragments of group m+1 are read (of group 0 of the next step at the end, once its rows have
  // landed), the stage rows of group m - their fragments are in registers - are refilled with the rows of the
  // step after next, one of the next step's weight fragments is read, and the indices four steps on and the
  // weight slice three steps on are requested.
  // SLOT = a % 2 is the stage being multiplied, wbuf = a % 3 the weight buffer whose fragments are in curW.
  // Returns true when the step was the last of its tile.
  int wbuf = 0;
  auto step = [&](int a, auto slotTag, F (&curW)[KK][NT], F (&nxtW)[KK][NT]) __attribute__((always_inline)) -> bool {
    constexpr int SLOT = decltype(slotTag)::value;
    // The two register sets alternate from group to group, across steps as well: with an odd number of groups
    // per step the set a group uses flips with the parity of the step (SLOT is that parity).
    constexpr int PAR = (MT & 1) ? SLOT : 0;
    constexpr int WREADS = (NQ + MT - 1) / MT;      // weight fragment reads per group
    // Loads ride behind MFMAs: the GPM gathers of a group behind its first GPM MFMAs, and the remaining
    // ("free") MFMA slots of the step, in order, carry the index load and then the WL weight loads.
    constexpr int FREE = NQ - GPM;                  // free slots per group
    static_assert(FREE >= 0 && MT * FREE >= 1 + WL, "a step has too few MFMAs to carry its loads");
    constexpr int freeBeforeWait = (MT - 1) * FREE; // free slots ahead of the wait (which opens the last group)
    constexpr int extraBeforeWait = (freeBeforeWait >= 1 ? IL : 0) +
                                    (freeBeforeWait - 1 > WL ? WL : (freeBeforeWait - 1 > 0 ? freeBeforeWait - 1 : 0));
    const bool lastOfTile = (ids[0] & kLastOfTile) != 0;
    const uint32_t partOff = chunkOff + ((ids[2] & ~kLastOfTile) % KS) * static_cast<uint32_t>(CS * ES);
    const int sW = static_cast<int>(ids[3] & ~kLastOfTile);
    const int nextBuf = wbuf + 1 == NWB ? 0 : wbuf + 1;
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      F(&cur)[KK] = rowBuf[(m + PAR) & 1];
      F(&nxt)[KK] = rowBuf[(m + 1 + PAR) & 1];
      int32_t(&ix)[GPM] = ixBuf[(m + PAR) & 1];
      if (m + 1 < MT) {
        readRowGroup(nxt, m + 1, SLOT);
        readIndex(a + 2, m + 1, ixBuf[(m + 1 + PAR) & 1]);
      } else {
        // everything issued before this step has landed: the rows of the next step, this wavefront's part of
        // the weight slice of the step after next, the indices of the step after that
        waitVmcnt<(MT - 1) * GPM + extraBeforeWait>();
        readRowGroup(nxt, 0, SLOT ^ 1);
        readIndex(a + 3, 0, ixBuf[(m + 1 + PAR) & 1]);
      }
#pragma unroll
      for (int e = m * WREADS; e < (m + 1) * WREADS && e < NQ; ++e)
        readWeight(nxtW, e, nextBuf);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int q = 0; q < NQ; ++q) {
        acc[m][q % NT] = Mfma<T>::k32(curW[q / NT][q % NT], cur[q / NT], acc[m][q % NT]);
        __builtin_amdgcn_sched_barrier(0);
        // the fragments of group m have left LDS (the MFMA above waited for them): refill its stage rows
        if (q < GPM) gatherOne(m * GPM + q, ix[q], partOff, SLOT);
        if (q >= GPM) {
          const int u = m * FREE + q - GPM;         // ordinal of this free slot within the step
          if (u == 0) ids[4] = loadIndex(a + 4);
          if (u >= 1 && u <= WL) weightLoad(u - 1, sW, wbuf);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    wbuf = nextBuf;
#pragma unroll
    for (int t = 0; t < 4; ++t) ids[t] = ids[t + 1];
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    return lastOfTile;
  };

  if constexpr (SPLIT > 1) {
    // the groups keep pace: the one with fewer steps meets the other's last barrier empty-handed
    for (int a = 0; a < mostSteps; a += 2) {
      if (a < mySteps) step(a, std::integral_constant<int, 0>{}, wtsA, wtsB);
      else __builtin_amdgcn_s_barrier();
      if (a + 1 >= mostSteps) break;
      if (a + 1 < mySteps) step(a + 1, std::integral_constant<int, 1>{}, wtsB, wtsA);
      else __builtin_amdgcn_s_barrier();
    }
    waitVmcnt<0>();                                 // loads issued for steps that do not exist: the stages are free
    if (group) {
#pragma unroll
      for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int n = 0; n < NT; ++n) reinterpret_cast<Acc*>(stage)[(m * NT + n) * 64 + lane] = acc[m][n];
    }
    __syncthreads();
    if (!group) {
      const Acc* const other = reinterpret_cast<const Acc*>(reinterpret_cast<const unsigned char*>(stage) +
                                                            NWB * WCH * 16 + WAVES * (2 * SLOTS * 16 + NI * WM * 4));
#pragma unroll
      for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int n = 0; n < NT; ++n) acc[m][n] += other[(m * NT + n) * 64 + lane];
      storeTile(firstPos);
    }
    __syncthreads();                                // the sums have been read: the next tile's rows may land
  } else {
  for (int a = 0;; a += 2) {
    if (step(a, std::integral_constant<int, 0>{}, wtsA, wtsB)) {
      storeTile(mulPos);
      if (++mulPos >= nMine) break;
    }
    if (step(a + 1, std::integral_constant<int, 1>{}, wtsB, wtsA)) {
      storeTile(mulPos);
      if (++mulPos >= nMine) break;
    }
  }
  }
  }
  waitVmcnt<0>();                                   // loads issued for steps that do not exist, and the stores
}

template <class T, int CIN, int COUT, int MT, int WAVES, int CO = COUT, bool DEAL = false, int SPLIT = 1>
__global__ void __launch_bounds__(64 * WAVES * SPLIT)
convPipe(const T* __restrict__ in, T* __restrict__ out, const T* __restrict__ wf, const float* __restrict__ bias,
         const float* __restrict__ requantM, const int32_t* __restrict__ nbr, int64_t nbrPitch, int tapMirror,
         const unsigned long long* __restrict__ tileMasks, int kVol, int64_t inRows, int64_t outRows, int relu,
         int xcdShift, const int32_t* __restrict__ numActOut, const int32_t* __restrict__ rowOrder) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  pipeTiles<T, CIN, COUT, MT, WAVES, CO, DEAL, SPLIT>(smem, in, out, wf, bias, requantM, nbr, nbrPitch, tapMirror, tileMasks, kVol, inRows, outRows,
                                     relu, xcdShift, numActOut, gridDim.x, rowOrder);
}

// The same with the tile chosen by the live rows (wavefronts of 32 rows: those of 48 take 278 registers, which workgroups of
// eight do not have); the host knows the capacity only.  Wavefronts past the tile's end at once.
template <class T, int CIN, int COUT>
__global__ void __launch_bounds__(512)
convPipeByRows(const T* __restrict__ in, T* __restrict__ out, const T* __restrict__ wf, const float* __restrict__ bias,
               const float* __restrict__ requantM, const int32_t* __restrict__ nbr, int64_t nbrPitch, int tapMirror,
               const unsigned long long* __restrict__ tileMasks, int kVol, int64_t inRows, int64_t outRows, int relu,
               int xcdShift, const int32_t* __restrict__ numActOut, int cus) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int tile = pipeTileRows(liveOutRows(numActOut, outRows), cus);
#define D3D_PIPE_BODY(WAVES)                                                                                            \
  {                                                                                                                     \
    if (wave >= WAVES) return;                                                                                          \
    pipeTiles<T, CIN, COUT, 2, WAVES>(smem, in, out, wf, bias, requantM, nbr, nbrPitch, tapMirror, tileMasks, kVol,     \
                                      inRows, outRows, relu, xcdShift, numActOut, gridDim.x);                           \
  }
  if (tile == 128) D3D_PIPE_BODY(4)
  else if (tile == 256) D3D_PIPE_BODY(8)
  else D3D_PIPE_BODY(6)
#undef D3D_PIPE_BODY
}

// 64 output channels: eight wavefronts of 64 rows, or of 48 where rounds of those tiles leave the CUs clearly less to do (with
// many rounds the wider tile is the better one whatever their number).
__host__ __device__ inline bool pipeTakes48(int64_t rows, int cus) {
  auto load = [&](int tile) { return (rows + static_cast<int64_t>(tile) * cus - 1) / (static_cast<int64_t>(tile) * cus) * tile; };
  return 10 * load(384) < 9 * load(512);
}
template <class T, int CIN, int COUT, bool DEAL>
__global__ void __launch_bounds__(512)
convPipeNarrowByRows(const T* __restrict__ in, T* __restrict__ out, const T* __restrict__ wf, const float* __restrict__ bias,
                     const float* __restrict__ requantM, const int32_t* __restrict__ nbr, int64_t nbrPitch, int tapMirror,
                     const unsigned long long* __restrict__ tileMasks, int kVol, int64_t inRows, int64_t outRows, int relu,
                     int xcdShift, const int32_t* __restrict__ numActOut, int cus) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  if (pipeTakes48(liveOutRows(numActOut, outRows), cus))
    pipeTiles<T, CIN, COUT, 3, 8>(smem, in, out, wf, bias, requantM, nbr, nbrPitch, tapMirror, tileMasks, kVol, inRows, outRows,
                                  relu, xcdShift, numActOut, gridDim.x);
  else
    pipeTiles<T, CIN, COUT, 4, 8, COUT, DEAL>(smem, in, out, wf, bias, requantM, nbr, nbrPitch, tapMirror, tileMasks, kVol, inRows, outRows,
                                              relu, xcdShift, numActOut, gridDim.x);
}

// LDS of a shape: three weight slices, two stages and four steps of indices per wavefront.
template <class T, int CIN, int COUT>
constexpr size_t pipeLds(int mt, int waves) {
  const int cs = CIN * static_cast<int>(sizeof(T)) > 128 ? 128 / static_cast<int>(sizeof(T)) : CIN;
  return static_cast<size_t>(3) * cs * COUT * sizeof(T) + static_cast<size_t>(waves) * (2 * 16 * mt * cs * sizeof(T) + 4 * 16 * mt * 4);
}

// 32-bit buffer offsets, and the 64 bits of a tap mask
inline bool pipeTakes(const ConvArgs& a, int64_t pitch, size_t rowBytes, int tileRows) {
  return a.kVol <= 64 && static_cast<uint64_t>(a.inRows) * rowBytes < 0xFFFF0000ull &&
         static_cast<uint64_t>(a.kVol) * static_cast<uint64_t>(pitch) * 4 < 0xFFFF0000ull &&
         static_cast<uint64_t>(a.outRows) + tileRows < 0x3FFFFFFFull;
}

template <class T, int CIN, int COUT, bool DEAL>
constexpr auto pipeByRowsKernel() {
  if constexpr (COUT < 128) return &convPipeNarrowByRows<T, CIN, COUT, DEAL>;
  else return &convPipeByRows<T, CIN, COUT>;
}

template <class T, int CIN, int COUT, bool DEAL = false>
int32_t launchPipeByRows(const ConvArgs& a, hipStream_t stream) {
  constexpr bool NARROW = COUT < 128;
  constexpr auto kernel = pipeByRowsKernel<T, CIN, COUT, DEAL>();
  const int64_t pitch = a.nbrPitch > 0 ? a.nbrPitch : a.outRows;
  if (!pipeTakes(a, pitch, CIN * sizeof(T), 512)) return D3D_ERR_UNSUPPORTED;
  constexpr size_t lds = pipeLds<T, CIN, COUT>(NARROW ? 4 : 2, 8);
  static_assert(lds <= kLdsLimit, "every shape fits a CU");
  static std::atomic<size_t> granted{64 * 1024};
  const int32_t rc = grantLds(kernel, lds, &granted);
  if (rc != D3D_OK) return rc;
  const ChipLayout chip = chipLayout();
  const int nXcd = 1 << chip.xcdShift, cus = chip.cus / nXcd * nXcd, perCu = kLdsLimit / lds > 1 ? 2 : 1;
  hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(cus * perCu)), dim3(512), lds, stream,
                     static_cast<const T*>(a.in), static_cast<T*>(a.out), static_cast<const T*>(a.weightsMfma), a.bias,
                     a.requantM, a.nbr, pitch, a.tapMirror, a.tileMasks, a.kVol, a.inRows, a.outRows, a.relu, chip.xcdShift,
                     a.numActOut, cus);
  return D3D_OK;
}

template <class T, int CIN, int COUT, int MT, int WAVES, int CO = COUT, int SPLIT = 1>
int32_t launchPipeCfg(const ConvArgs& a, hipStream_t stream) {
  constexpr int TM = 16 * MT * WAVES, COLS = COUT / CO;
  constexpr size_t lds = SPLIT * pipeLds<T, CIN, CO>(MT, WAVES);
  const int64_t pitch = a.nbrPitch > 0 ? a.nbrPitch : a.outRows;
  if (lds > kLdsLimit || !pipeTakes(a, pitch, CIN * sizeof(T), TM)) return D3D_ERR_UNSUPPORTED;
  const int tiles = static_cast<int>((a.outRows + TM - 1) / TM);
  // persistent workgroups: as many as the CUs can hold at this LDS footprint, never more than there are tiles (three where
  // they fit: int8 64 -> 64 127 us with two, 121 with three on 1.07 million rows, 31 and 28 on 190 000; fp16 32 -> 64 153 and
  // 147, 28.7 and 26)
  int perCu = static_cast<int>(kLdsLimit / lds);
  if (perCu > 3) perCu = 3;
  if (perCu < 1) perCu = 1;
  const ChipLayout chip = chipLayout();
  const int nXcd = 1 << chip.xcdShift;
  int blocks = (tiles + nXcd - 1) / nXcd * nXcd * COLS;
  const int most = chip.cus * perCu / (nXcd * COLS) * (nXcd * COLS);
  if (blocks > most) blocks = most;
  auto launch = [&](auto kernel, std::atomic<size_t>* granted) -> int32_t {
    const int32_t rc = grantLds(kernel, lds, granted);
    if (rc != D3D_OK) return rc;
    hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(blocks)), dim3(64 * WAVES * SPLIT), lds, stream, static_cast<const T*>(a.in),
                       static_cast<T*>(a.out), static_cast<const T*>(a.weightsMfma), a.bias, a.requantM, a.nbr, pitch, a.tapMirror,
                       a.tileMasks, a.kVol, a.inRows, a.outRows, a.relu, chip.xcdShift, a.numActOut, a.rowOrder);
    return D3D_OK;
  };
  static std::atomic<size_t> granted{64 * 1024};
  // an instantiation of its own: the list costs the others registers they use (260 000 rows, 64 -> 64: 1 % of a pass).  Two-byte
  // tiles of 32-row wavefronts are for few rows and never get there; which types gain: see TileDeal
  if constexpr (SPLIT == 1 && (sizeof(T) == 4 || (sizeof(T) == 2 && CIN >= 64 && MT > 2))) {
    static std::atomic<size_t> grantedDeal{64 * 1024};
    if (a.rowOrder || (a.tileMasks && tiles > (sizeof(T) == 4 ? 1 : kDealRounds) * (blocks / COLS)))
      return launch(&convPipe<T, CIN, COUT, MT, WAVES, CO, true>, &grantedDeal);
  }
  if (a.rowOrder) {
    setError("conv: a tile shape that does not take rows in another order");
    return D3D_ERR_DEVICE;
  }
  return launch(&convPipe<T, CIN, COUT, MT, WAVES, CO, false, SPLIT>, &granted);
}

// Configuration per layer shape, measured on the layers of a VoxelNet backbone (120k voxels): rows per wavefront
// 16 * MT, wavefronts per workgroup.  64 x 64 and narrower tiles afford 8 wavefronts (4 wavefronts of 128 rows,
// which read half the weight fragments per MFMA, measured slower on a 64 -> 64 layer: 68 us against 58 - one
// wavefront per SIMD has nobody to hide its waits); 128 output channels double the accumulators, so the wavefront
// tile halves.  32 -> 32 (more taps than conv_solo.h keeps resident) takes 8
// wavefronts as well (two workgroups of 78 KB per CU): with 27 taps 38 us against 41 with 4, 40 with three
// 4-wavefront workgroups per CU, 41 with 128-row and 42 with 48-row wavefront tiles.  Two taps per step
// (a stage row holding the neighbours under two taps side by side, the step of a 64-channel layer) measured slower
// on 32 -> 64 in every tile shape tried (45-57 us against 36): the stage doubles, one workgroup fits a CU instead of
// two, and the layer needs the wavefronts more than the longer steps.
// Layers of 128 output channels pick the shape by the row count: the time of a layer that fits one round is that of ONE
// tile.
template <class T, int CIN, int COUT>
int32_t launchPipeShape(const ConvArgs& a, hipStream_t stream) {
  // shapes go by the bytes of an input row (the stage) and by the output channels (the accumulators): an int8 layer
  // takes the shape of the two-byte layer with half its input channels
  constexpr int RB = CIN * static_cast<int>(sizeof(T));
  // rows in the order of their taps: the narrower a tile, the fewer taps it has
  if constexpr (sizeof(T) == 2 && COUT == 128 && CIN >= 64)
    if (a.rowOrder) return launchPipeCfg<T, CIN, COUT, 3, 4, 64>(a, stream);
  if constexpr (sizeof(T) == 4) {
    // fp32: a step's MFMAs take eight times the cycles of a two-byte step with the same bytes, so the matrix pipe is
    // the bound and the tile only has to spread over the CUs: 128 rows, two or three workgroups per CU (16 -> 128: eight
    // wavefronts).  64 -> 64 with 150 000 rows runs at 130 TFLOP/s of issued MFMAs against the 157 of the pipe (630 us on
    // the vector kernel); skipping a 16-row group's MFMAs when none of its rows has the tap gained 15-20 us on strided and
    // inverse layers and cost as much on the dense ones: the barrier waits for the fullest group either way
    // Layers of 64 and 128 output channels share a tile's channels out to workgroups of 32: with the matrix pipe as the bound
    // a layer's time goes by the workgroups of the fullest CU, and smaller ones spread more evenly.  us with all channels /
    // shared out: 64 -> 64, 30 000 rows 64 / 61, 118 000 212 / 203, 144 000 (4.4 tiles of all channels to a CU) 260 / 238,
    // 261 000 402 / 398; 32 -> 64, 262 000 rows 208 / 207; 128 -> 128, 17 000 rows 409 / 163, 40 000 (a 256-row tile of all channels on
    // 156 of 256 CUs) 409 / 274, 47 500 410 / 324
    if constexpr (COUT >= 64 && CIN >= 32) return launchPipeCfg<T, CIN, COUT, 2, 4, 32>(a, stream);
    else if constexpr (COUT >= 128) return launchPipeCfg<T, CIN, COUT, 2, 8>(a, stream);
    else return launchPipeCfg<T, CIN, COUT, 2, 4>(a, stream);
  } else if constexpr (RB == 128 && COUT == 64) {
    // 512- or 384-row tiles; few rows take the smallest of 128, 256 and 512 whose tiles still fit one round of the CUs (64 -> 64:
    // 15 600 rows 16 us against 25 with 512-row tiles, 43 000 rows 19 against 26; with 118 000 rows, more than one round
    // of 256-row tiles, those take 35 against 30)
    if constexpr (sizeof(T) == 2) {
      const int64_t cus = chipLayout().cus;
      // up to 192 rows per CU the steps of a tile are shared by two groups of wavefronts: one group of four leaves LDS reads and
      // MFMAs of a SIMD's only wavefront to take turns.  43 000 rows 17.3 -> 15.4 us (256-row tiles on 169 CUs before)
      if (a.outRows <= 128 * cus) return launchPipeCfg<T, CIN, COUT, 2, 4, 64, 2>(a, stream);
      if (a.outRows <= 192 * cus) return launchPipeCfg<T, CIN, COUT, 3, 4, 64, 2>(a, stream);
      if (a.outRows <= 256 * cus) return launchPipeCfg<T, CIN, COUT, 2, 8>(a, stream);
      // 384-row tiles by the live rows: 196 000 rows, one and a half rounds of 512, two of 384, 52 -> 46 us; 262 000, two
      // rounds of 512, stay at 60 (64 with 384).  Capacities whose 512-row tiles may be dealt choose as well: with room for 600 000
      // rows 196 000 live ones take 58 us, 280 000 74, and 64 and 85 in 512-row tiles
      if (a.tileMasks && a.outRows > kDealRounds * 512 * cus) return launchPipeByRows<T, CIN, COUT, true>(a, stream);
      return launchPipeByRows<T, CIN, COUT>(a, stream);
    } else {
      return launchPipeCfg<T, CIN, COUT, 4, 8>(a, stream);
    }
  } else if constexpr (COUT >= 128) {
    const int64_t cus = chipLayout().cus;
    // D3D_CONV_PIPE_SHAPE=rows,wavefronts (tests): a shape the layer has whatever the rows (rows per wavefront); others, and
    // what the kernels choose by the live rows, are not forced
    const char* const env = debugEnv("D3D_CONV_PIPE_SHAPE");
    auto forced = [&](const char* shape) { return env && std::strcmp(env, shape) == 0; };
    if constexpr (sizeof(T) == 1 || CIN >= 64) {
      // One workgroup of four wavefronts per CU that takes all 128 channels adds the time of its LDS reads (each wavefront
      // reads a step's whole weight slice) to that of its MFMAs: without MFMAs, gathers and weight loads a 24 000-row layer
      // still took 21 of 34 us.  So a tile's channels are shared out to workgroups of 64 (with few rows, 32): two workgroups
      // of half the slices fit a CU and each computes while the other reads.  us of 128 -> 128 and of 64 -> 128 with all
      // channels / shared out, fp16: 11 000 rows 33 / 22 and 22 / 15, 17 500 rows 31 / 25.5 and 20 / 17, 23 500 rows 32 / 27
      // and 23 / 18, 40 000 rows 42 / 41 and 29.5 / 26, 47 500 rows 44 / 43.5 and 29 / 28, 95 000 rows 87 / 73 and 54.5 / 48,
      // 188 000 rows 127 / 134 and 87 / 85.5 (the three-tap column layer behind it 32 / 26); int8: 22.5 / 16 and 17 / 13.5, 21 / 17
      // and 15 / 13.5, 21 / 18 and 18 / 14, 26 / 24.5 and 21.5 / 18.5, 27.5 / 25.5 and 20 / 20, 50 / 42 and 28.5 / 34, 87 / 79 and
      // 51 / 57.  From 188 000 rows on 128 -> 128 gives back 5 % in two-byte types, and 64 -> 128 a tenth in int8: over the layers
      // of a network (two of the one, one of the other and a column layer) as much is won, so no further line is drawn.
      // The wider tile wins where it fits as many workgroups to a CU: the lines are whole rounds of one and of two per CU.
      const bool shared4 = forced("32,4"), shared3 = forced("48,4"), free = !shared4 && !shared3;
      if constexpr (RB >= 128) {
        // one workgroup per CU: its steps are shared by two groups of wavefronts (128 -> 128, 23 000 rows: fp16 25.8 -> 23.1 us,
        // int8 17.5 -> 15.5; a pass of 9 000 voxels in fp16 267 -> 256 with the 64 -> 64 layers).  Bound by LDS: 60 KB of fragments
        // and rows a step, 25 000 clocks of them in all.
        if (free && a.outRows <= 32 * cus) return launchPipeCfg<T, CIN, COUT, 2, 4, 32, 2>(a, stream);
        if (free && a.outRows <= 64 * cus) return launchPipeCfg<T, CIN, COUT, 2, 4, 64, 2>(a, stream);
        if (free && a.outRows <= 96 * cus) return launchPipeCfg<T, CIN, COUT, 3, 4, 64, 2>(a, stream);
      }
      if (free && a.outRows <= 32 * cus) return launchPipeCfg<T, CIN, COUT, 2, 4, 32>(a, stream);   // 29 -> 18 us
      if (shared4 || (free && (a.outRows <= 64 * cus || (a.outRows > 96 * cus && a.outRows <= 128 * cus))))
        return launchPipeCfg<T, CIN, COUT, 2, 4, 64>(a, stream);
      // Past one round of two 192-row workgroups per CU (49 152 rows) a few of them have a second tile, 50 000 live rows take
      // 61 us, 55 000 70, where 256-row tiles of all channels take 52 and 53: up to 288 rows per CU the two-byte layers choose
      // by the live rows.  The line is drawn at the capacity, six percent above the round, since a capacity is above its live
      // rows, and that suits one head-room: 47 500 live rows take 44 us under the line and 51 above it (capacities of 1.25 and
      // 1.5 times, where the shared-out tile would take 45), 50 000 live rows below the line take the 61.  The kernel that
      // chooses on the device does not hold the shared-out shape.
      if constexpr (sizeof(T) > 1)
        if (free && a.outRows > 204 * cus && a.outRows <= 288 * cus) return launchPipeByRows<T, CIN, COUT>(a, stream);
      return launchPipeCfg<T, CIN, COUT, 3, 4, 64>(a, stream);
    } else {
      // 32 -> 128: one round of the smallest tile that has one (128 or 256 rows in wavefronts of 32, 192 in wavefronts of 48);
      // beyond, the tile that loads the busiest CU least, by the live rows
      const bool rows128 = forced("32,4"), rows192 = forced("48,4"), rows256 = forced("32,8"), free = !rows128 && !rows192 && !rows256;
      if (rows128 || (free && a.outRows <= 128 * cus)) return launchPipeCfg<T, CIN, COUT, 2, 4>(a, stream);
      if (rows192 || (free && a.outRows <= 192 * cus)) return launchPipeCfg<T, CIN, COUT, 3, 4>(a, stream);
      if (rows256 || (free && a.outRows <= 256 * cus)) return launchPipeCfg<T, CIN, COUT, 2, 8>(a, stream);
      return launchPipeByRows<T, CIN, COUT>(a, stream);
    }
  } else if constexpr (RB == 64 && COUT == 32) {
    return launchPipeCfg<T, CIN, COUT, 4, 8>(a, stream);
  } else {
    // 256-row tiles; 128-row ones while those fit the two workgroups that a CU holds (32 -> 64: 15 600 rows 12.7 us
    // against 15.7, 43 000 rows 14.4 against 16.4, but 118 000 rows, nearly four per CU, 26 against 21)
    if constexpr (sizeof(T) == 2 && CIN == 32 && COUT == 64)
      if (a.outRows <= 256 * static_cast<int64_t>(chipLayout().cus)) return launchPipeCfg<T, CIN, COUT, 2, 4>(a, stream);
    return launchPipeCfg<T, CIN, COUT, 4, 4>(a, stream);
  }
}

template <class T>
int32_t launchPipe(const ConvArgs& a, hipStream_t stream) {
#define D3D_PIPE_CASE(CI, CO) \
  if (a.cin == CI && a.cout == CO) return launchPipeShape<T, CI, CO>(a, stream);
  if constexpr (sizeof(T) == 4) {
    D3D_PIPE_CASE(16, 64)
    D3D_PIPE_CASE(16, 128)
  }
  if constexpr (sizeof(T) >= 2) {  // rows of 64 bytes at least
    D3D_PIPE_CASE(32, 32)
    D3D_PIPE_CASE(32, 64)
    D3D_PIPE_CASE(32, 128)
  }
  D3D_PIPE_CASE(64, 32)
  D3D_PIPE_CASE(64, 64)
  D3D_PIPE_CASE(64, 128)
  D3D_PIPE_CASE(128, 32)
  D3D_PIPE_CASE(128, 64)
  D3D_PIPE_CASE(128, 128)
#undef D3D_PIPE_CASE
  return D3D_ERR_UNSUPPORTED;
}

}  // namespace convk
}  // namespace d3d
