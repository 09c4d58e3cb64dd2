// Hand-written gfx950 kernels for decision-forest inference.
//
// They replace the kernels the reference generates from its schedules
// (src/gpu/GPUSchedules.cpp, src/mlir/CodeGenStateMachine.cpp:149-243 scalar
// tile step, src/mlir/WalkDecisionTreeLoweringPass.cpp:23-110 walk loops,
// src/gpu/GPURepresentations.cpp:279-399 row caching, src/mlir/LowerReduceOps.cpp
// :119-187 and :921-1003 reductions, src/mlir/LowerToMidLevelIR.cpp:554-648
// result initialisation and sigmoid).
#include "kernels.h"

#include <hip/hip_ext.h>

#include <algorithm>
#include <atomic>
#include <cmath>

namespace tbamd {

namespace {

__device__ __forceinline__ float AsFloat(uint32_t u) { return __uint_as_float(u); }

// LDS reads by absolute LDS address.  The kernels below use dynamic LDS only,
// which the compiler places at LDS address 0, so an offset into the dynamic
// array is the address itself and no base has to be added per access.
typedef uint32_t U32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t U32x4 __attribute__((ext_vector_type(4)));
typedef const __attribute__((address_space(3))) U32x2 *LdsNodePtr;
typedef const __attribute__((address_space(3))) float *LdsFloatPtr;
__device__ __forceinline__ U32x2 LdsLoadNode(uint32_t address) { return *(LdsNodePtr)(uintptr_t)address; }
__device__ __forceinline__ float LdsLoadFloat(uint32_t address) { return *(LdsFloatPtr)(uintptr_t)address; }
typedef const __attribute__((address_space(3))) uint8_t *LdsBytePtr;
__device__ __forceinline__ uint32_t LdsLoadByte(uint32_t address) { return *(LdsBytePtr)(uintptr_t)address; }
typedef const __attribute__((address_space(3))) uint16_t *LdsHalfPtr;
__device__ __forceinline__ uint32_t LdsLoadHalf(uint32_t address) { return *(LdsHalfPtr)(uintptr_t)address; }

// A node's child pointer (the low half of its meta word) plus `more`: a 16-bit addition leaves the upper half of the result zero and
// takes 2.2 cycles of a SIMD that eight waves share (2.5: four), where one that selects a half (SDWA) or a compare takes 4.1 to 4.4.
__device__ __forceinline__ uint32_t AddChild(uint32_t meta, uint32_t more) {
  uint32_t address;
  asm("v_add_u16_e32 %0, %1, %2" : "=v"(address) : "v"(meta), "v"(more));
  return address;
}

// How a node's 16-bit feature offset addresses the row tile of the row-parallel kernel.
enum RowTileMode : int {
  kTileF32Bytes = 0, // f32 tile, offset in bytes
  kTileF32Words = 1, // f32 tile, offset in units of 4 bytes (tiles above 64 KB)
  kTileRankU8 = 2,   // one-byte rank tile (rank-quantised rows), offset in units of 4 bytes
  kTileRankU16 = 3   // two-byte rank tile [feature pair][row][2], offset in bytes
};
constexpr bool IsRankTile(int mode) { return mode == kTileRankU8 || mode == kTileRankU16; }

// A rank tile's comparison: the row's rank among the feature's thresholds against the node's threshold index.
template <int kMode>
__device__ __forceinline__ bool RankGoesLeft(uint32_t address, uint32_t thresholdIndex) {
  return (kMode == kTileRankU8 ? LdsLoadByte(address) : LdsLoadHalf(address)) <= thresholdIndex;
}


// Copies the block's rows (contiguous, row-major in global memory) into LDS.  Loads are 16-byte wide (dword alignment is
// enough for the hardware), issued several at a time per lane and unconditional, their places clamped into the live part of
// the batch, so that they overlap; nothing outside the batch is touched.
constexpr int kStageUnroll = 8;
typedef float StagePiece __attribute__((ext_vector_type(4), aligned(4)));

// ... transposed, tile[f * R + r] (R: a multiple of 64).  A wave takes 16 rows x 4 pieces of 4 features: 64 bytes of a row
// per cache line touched, and of the 64 lanes that write a feature's value 4 meet in a bank.  (A wave along a row, as for
// the copy as it stands, makes 16-way conflicts at 64 features and 32-way ones at 128.)  Rows past the end are copies of the
// last one.  Walk kernels, before and after: 50001 rows x 90 features, 100 trees 24.0 -> 19.6 us; 300000 x 150, 300 trees
// 191 -> 144; 100000 x 300, 100 trees 83 -> 50; 2^20 x 90, 800 deep trees 1266 -> 1204; 2^20 x 28, 1000 trees 1156 -> 1149.
__device__ __forceinline__ void StageRowsTransposed(const float *__restrict__ src, int valid, int R, int F, float *tile, int tid,
                                                    int threads) {
  if (valid < 1) return;
  if (F < 4) {
    for (int e = tid; e < valid * F; e += threads) {
      const int r = e / F;
      tile[(e - r * F) * R + r] = src[e];
    }
    return;
  }
  constexpr int kUnroll = 4;
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), waves = threads >> 6;
  const int shift = F > 12 ? 4 : 5;                             // lanes along the rows (log2), the others along the pieces
  const int across = 64 >> shift, groups = ((F + 3) / 4 + across - 1) / across;
  const int rowGroups = R >> shift, rowWaves = rowGroups < waves ? rowGroups : waves, acrossWaves = waves / rowWaves;
  const int firstGroup = wave / rowWaves;
  if (firstGroup >= acrossWaves) return;                        // (a number of waves that does not divide)
  for (int rg = wave - firstGroup * rowWaves; rg < rowGroups; rg += rowWaves) {
    const int r = rg << shift | (lane & ((1 << shift) - 1));
    const float *row = src + (r < valid ? r : valid - 1) * F;
    for (int g = firstGroup; g < groups; g += acrossWaves * kUnroll) {
      StagePiece v[kUnroll];
      int f[kUnroll];
#pragma unroll
      for (int u = 0; u < kUnroll; ++u) {
        // (the last pieces overlap, or repeat, the one before: the same values in the same places)
        f[u] = ((g + u * acrossWaves) * across + (lane >> shift)) * 4;
        f[u] = f[u] < F - 4 ? f[u] : F - 4;
        v[u] = *reinterpret_cast<const StagePiece *>(row + f[u]);
      }
#pragma unroll
      for (int u = 0; u < kUnroll; ++u) {
        if (g + u * acrossWaves >= groups) break;
#pragma unroll
        for (int j = 0; j < 4; ++j) tile[(f[u] + j) * R + r] = v[u][j];
      }
    }
  }
}

// ... as they stand, tile[r * rowWords + f].  Rows past the end read as 0.
__device__ __forceinline__ void StageRows(const float *__restrict__ src, int valid, int R, int F, int rowWords, float *tile, int tid,
                                          int threads) {
  const int total = R * F;
  const int live = valid * F;
  const bool aligned = (reinterpret_cast<uintptr_t>(src) & 15u) == 0;
  const int vecs = aligned ? total >> 2 : 0;    // 16-byte pieces handled by the vector path
  const int liveVecs = aligned ? live >> 2 : 0; // pieces that lie entirely inside the batch
  const float invF = 1.0f / (float)F;
  typedef float F32x4 __attribute__((ext_vector_type(4)));
  const F32x4 *src4 = reinterpret_cast<const F32x4 *>(src);
  for (int base = 0; base < vecs; base += threads * kStageUnroll) {
    F32x4 v[kStageUnroll];
#pragma unroll
    for (int u = 0; u < kStageUnroll; ++u) {
      const int idx = base + u * threads + tid;
      const int clamped = idx < liveVecs ? idx : (liveVecs > 0 ? liveVecs - 1 : 0);
      v[u] = liveVecs > 0 ? src4[clamped] : F32x4{0.f, 0.f, 0.f, 0.f};
    }
#pragma unroll
    for (int u = 0; u < kStageUnroll; ++u) {
      const int idx = base + u * threads + tid;
      if (idx >= vecs) continue;
      const int e0 = idx << 2;
      int r = (int)((float)e0 * invF);
      if (r * F > e0) --r;
      if ((r + 1) * F <= e0) ++r;
      int f = e0 - r * F;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int e = e0 + j;
        // elements of the one partially live piece are left to the scalar tail below
        if (idx < liveVecs || e >= live) {
          const float value = idx < liveVecs ? v[u][j] : 0.0f;
          tile[r * rowWords + f] = value;
        }
        if (++f == F) { f = 0; ++r; }
      }
    }
  }
  // scalar: the live elements of the partially live piece, which the vector path skipped ...
  const int skippedEnd = live < (vecs << 2) ? live : (vecs << 2);
  for (int e = (liveVecs << 2) + tid; e < skippedEnd; e += threads) {
    const int r = e / F;
    const int f = e - r * F;
    tile[r * rowWords + f] = src[e];
  }
  // ... and whatever lies behind the last whole 16-byte piece (everything, for unaligned input)
  for (int e = (vecs << 2) + tid; e < total; e += threads) {
    const int r = e / F;
    const int f = e - r * F;
    const float value = e < live ? src[e] : 0.0f;
    tile[r * rowWords + f] = value;
  }
}

// ---------------------------------------------------------------------------
// Row-parallel walk.  The block owns `rowsPerBlock` rows, kept transposed in
// LDS (feature-major) so that lane i always reads bank i%64 no matter which
// feature its node tests.  Trees are streamed through LDS one group at a time:
// either the next group is fetched into registers while the current one is walked
// (PF > 0), or the group is copied by direct global-to-LDS loads between the two
// barriers of its round while the compute unit's other blocks walk (PF == 0).
// A lane walks K trees at a time in lock step: all lanes take `depth` steps and
// leaves hold the walk in place (see device_model.h), so the loop body has no
// leaf test and no divergence.  Where leaves stay out of the groups (kWalkOutside) their values are gathered from L2,
// asked for when a bundle ends and added when the next one does: 16 address cycles per wave and tree on a path the walk
// leaves idle, for two cycles of the LDS pipe and 20 to 50 % of a group's room (2^20 rows x 28 features, 1000 trees of
// depth 8 1162 -> 1069 us; conflicts 0.28 -> 0.16 cycles an LDS instruction, LDS pipes 83 -> 81 % and VALUs 81 -> 90 % busy, the last with the
// additions above too).  `treeThreads` lanes (in different waves) share
// one row and split each group's bundles between them, which buys occupancy
// without growing the row tile; their sums meet in an LDS cross-wave pass.
// Sums are kept in double; trees are added in packed order.
// ---------------------------------------------------------------------------
// kDefer (peeled walks, src/mlir/ProbabilityBasedTilingTransform.cpp:66-73, src/mlir/WalkDecisionTreeLoweringPass.cpp
// :231-315, the way this hardware wants them): the lock-step walk of a tree stops at the level a hit-count
// profile says it still pays (device_model.h: stubs).  A row that ends on a stub is queued by its wave as
// (row, tail node); whenever 64 entries have come together - whatever trees they belong to - the wave walks
// them on densely, one entry per lane, to their leaves, and hands the leaf values back to the rows' lanes
// through LDS.  The subtrees below the stubs are not part of the tree groups: the dense walk reads its nodes
// from global memory (they stay in L2), so the queue outlives the groups and is emptied once more at the end.
// Lock step spends its LDS reads on all 64 rows of a wave even when three of them still move; the queue spends
// 64 lanes on 64 rows that do, its node reads go through the vector memory path, which the walk leaves idle,
// and only its feature reads (at scattered addresses now) come out of LDS.
//
// kVariant picks what is compiled in beside the plain walk (each costs the plain walk about a percent when it
// is merely present): kWalkDump the leaf-id dump of the parity checks, kWalkDefer the deferred tails, kWalkFuse
// the classifiers' running arg-max (WalkScalars::fuseArgmax), kWalkOwn and kWalkOwnFuse classes of the tree threads' own
// (WalkScalars::ownClasses; as a run-time branch of the plain walk it cost 1000 trees without classes 40 %: SGPRs).
// kWalkOutside is added to those (not to the dump, which looks where the leaves are, nor to deferred tails) where the leaves of a
// bundle's last level stay in global memory (PackedModel::leavesOutside): the walk's last step leads to their place, their values
// are asked for there and added a bundle later.  (As a run-time branch it cost 1000 trees on 2^20 rows 2 %.)
enum WalkVariant : int { kWalkPlain = 0, kWalkDump = 1, kWalkDefer = 2, kWalkFuse = 3, kWalkOwn = 4, kWalkOwnFuse = 5, kWalkOutside = 8 };

// Groups [gBegin, gEnd) of one row block: everything a block of the row-parallel walk does.  `slice` names the slot of
// the partial sums this part fills.
template <int K, int PF, int kMode, int kVariantBits>
__device__ __forceinline__ void
WalkRowBlock(unsigned char *lds, int64_t rowBlock, int gBegin, int gEnd, int slice,
             const float *__restrict__ x, const uint4 *__restrict__ nodes16,
             const DeviceBundle *__restrict__ bundles, const DeviceNode *__restrict__ bundleRoots,
             const DeviceGroup *__restrict__ groups,
             const WalkScalars &s, float *__restrict__ out, int8_t *__restrict__ classOut,
             double *__restrict__ partial, int32_t *__restrict__ leafIds, const int32_t *__restrict__ nodeOrigin,
             const int32_t *__restrict__ slotTree, const U32x2 *__restrict__ tailNodes, const int32_t *__restrict__ tailOrigin) {
  constexpr int kVariant = kVariantBits & ~kWalkOutside;
  constexpr bool kDump = kVariant == kWalkDump, kDefer = kVariant == kWalkDefer, kOutside = (kVariantBits & kWalkOutside) != 0;
  constexpr bool kFuse = kVariant == kWalkFuse || kVariant == kWalkOwnFuse;
  const bool own = kVariant == kWalkOwn || kVariant == kWalkOwnFuse || (kDump && s.ownClasses);
  // LDS: [tree group nodes | transposed row tile].  The group sits at LDS
  // address 0 so that node pointers are LDS addresses as stored.
  const int tid = threadIdx.x;
  const int threads = blockDim.x;
  const int RB = s.rowsPerBlock;
  const int TT = s.treeThreads;
  const int lane = tid & (RB - 1);
  // uniform inside a wave (RB is a multiple of 64); readfirstlane tells the compiler so
  const int tt = __builtin_amdgcn_readfirstlane(tid / RB);
  const int F = s.numFeatures;
  const int64_t row0 = rowBlock * RB;
  const int64_t remaining = s.rows - row0;
  const int valid = remaining < RB ? (int)remaining : RB;

  // Direct staging: a group is copied by global -> LDS loads (lane i of a wave-wide load leaves its 16 bytes at base +
  // 16 i, lanes switched off write nothing): no staging registers, no LDS store instructions.  The block waits for its
  // own copy; the CU's other block walks meanwhile, which is why launch plans ask for this form only when two blocks
  // fit a CU.
#define TBAMD_COPY_GROUP(GRP)                                                                                          \
  {                                                                                                                    \
    const U32x4 *src = reinterpret_cast<const U32x4 *>(nodes16) + ((GRP).nodeBegin >> 1);                              \
    const int pieces = (int)((GRP).nodeCount >> 1);                                                                    \
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);                                                         \
    for (int first = wave * 64; first < pieces; first += threads)                                                      \
      if (first + (tid & 63) < pieces)                                                                                 \
        __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)(src + first + (tid & 63)),   \
                                         (__attribute__((address_space(3))) void *)(lds + (uint32_t)first * 16u), 16, 0, 0); \
  }
  // the first group is on its way while the rows are staged
  if (PF == 0 && gBegin < gEnd) TBAMD_COPY_GROUP(groups[gBegin])

  uint32_t column; // LDS address of this row's feature 0
  if (IsRankTile(kMode)) {
    // Ranks arrive already tiled: plain copy.  One byte each as [row block][feature][row] (the pad feature's
    // column is filled here), or two bytes each as [row block][feature pair][row][2], pad feature included.
    typedef uint32_t Piece __attribute__((ext_vector_type(4)));
    const int tileBytes = kMode == kTileRankU8 ? F * RB : ((F + 2) >> 1) * RB * 4;
    const Piece *src = reinterpret_cast<const Piece *>(reinterpret_cast<const uint8_t *>(x) + rowBlock * tileBytes);
    Piece *dst = reinterpret_cast<Piece *>(lds + s.groupRegionBytes);
    const int pieces = tileBytes >> 4;
    for (int base = 0; base < pieces; base += threads * kStageUnroll) {
      Piece v[kStageUnroll];
#pragma unroll
      for (int u = 0; u < kStageUnroll; ++u) {
        const int idx = base + u * threads + tid;
        v[u] = src[idx < pieces ? idx : pieces - 1];
      }
#pragma unroll
      for (int u = 0; u < kStageUnroll; ++u) {
        const int idx = base + u * threads + tid;
        if (idx < pieces) dst[idx] = v[u];
      }
    }
    if (kMode == kTileRankU8) {
      for (int i = tid; i < RB; i += threads) lds[s.groupRegionBytes + (uint32_t)F * RB + i] = 0; // pad feature: rank 0
      column = s.groupRegionBytes + (uint32_t)lane;
    } else {
      column = s.groupRegionBytes + (uint32_t)lane * 4u;
    }
  } else {
    float *rowTile = reinterpret_cast<float *>(lds + s.groupRegionBytes);
    // Stage the block's rows: coalesced reads of the contiguous row-major tile, transposed writes.
    StageRowsTransposed(x + row0 * F, valid, RB, F, rowTile, tid, threads);
    for (int i = tid; i < RB; i += threads) rowTile[F * RB + i] = -INFINITY; // pad feature: keeps leaves in place
    column = s.groupRegionBytes + (uint32_t)lane * 4u;
  }
  // Deferred tails: the wave's queue of (row, node) entries, 128 of 4 bytes behind the row tile; while the wave
  // walks 64 of them on, the same 512 bytes take the leaf values on their way back (a double per lane).
  const uint32_t queueAddress = ((s.groupRegionBytes + (uint32_t)(F + 1) * RB * 4u + 15u) & ~15u) +
                                (uint32_t)__builtin_amdgcn_readfirstlane(tid >> 6) * kDeferBytesPerWave;
  uint32_t *queue = reinterpret_cast<uint32_t *>(lds + queueAddress);
  double *handBack = reinterpret_cast<double *>(lds + queueAddress);
  const uint32_t waveColumn = column - (uint32_t)(tid & 63) * 4u; // LDS address of feature 0 of the wave's first row
  const uint32_t laneTag = (uint32_t)(tid & 63) << 26;            // a queue entry: lane << 26 | tail index
  uint32_t queued = 0;                                            // entries in the queue (the same in every lane)

  const int C = s.numClasses;
  const int64_t row = row0 + lane;
  double *partialRow = partial ? partial + ((int64_t)slice * s.rows + row) * (C > 0 ? C : 1) : nullptr;
  // LDS cross-wave pass: the tree threads of a row leave their sums here and tree thread 0 adds
  // them in thread order.  Classifiers meet at class boundaries, while a tree group is live, so
  // their meeting area sits behind the row tile; otherwise the (then idle) group region is used.
  double *meet = reinterpret_cast<double *>(
      C > 0 && !own ? lds + ((s.groupRegionBytes + (kMode == kTileRankU16 ? (uint32_t)((F + 2) >> 1) * RB * 4u
                                                                  : (uint32_t)(F + 1) * RB * (kMode == kTileRankU8 ? 1u : 4u)) + 7u) & ~7u)
            : lds);

  double acc = 0.0;
  float leaf[K]; // kOutside: the last bundle's leaf values, on their way
#pragma unroll
  for (int k = 0; k < K; ++k) leaf[k] = 0.0f;
#define TBAMD_ADD_LEAVES                                                                                               \
  if (kOutside) {                                                                                                      \
    _Pragma("unroll") for (int k = 0; k < K; ++k) {                                                                    \
      acc += (double)leaf[k];                                                                                          \
      leaf[k] = 0.0f;                                                                                                  \
    }                                                                                                                  \
  }
  int curClass = own ? tt : 0;
  float best = -INFINITY; // fuseArgmax: running maximum of the class sums and its class (tree thread 0)
  int bestClass = 0;

  // Register double buffer for the next tree group.  Loads are unconditional
  // (index clamped) so that they stay in flight across the walk.  PF == 0 is the other way of staging: no
  // registers, the group goes straight from global memory into LDS between the two barriers (below).
  U32x4 fetched[PF > 0 ? PF : 1];
#define TBAMD_PREFETCH_GROUP(NEXTGRP)                                                                                  \
  {                                                                                                                    \
    const DeviceGroup nextGrp = (NEXTGRP);                                                                             \
    const U32x4 *src = reinterpret_cast<const U32x4 *>(nodes16) + (nextGrp.nodeBegin >> 1);                            \
    const int last = (int)(nextGrp.nodeCount >> 1) - 1;                                                                \
    _Pragma("unroll") for (int i = 0; i < PF; ++i) {                                                                   \
      const int idx = tid + i * threads;                                                                               \
      fetched[i] = src[idx < last ? idx : last];                                                                       \
    }                                                                                                                  \
  }
  // Ends class `curClass`: the row's tree threads meet in LDS and thread 0 stores the class sum.
  // Uniform across the block (class boundaries are bundle positions), so the barriers are safe.
#define TBAMD_FLUSH_CLASS(UPTO)                                                                                        \
  {                                                                                                                    \
    if (TT > 1) {                                                                                                      \
      __syncthreads();                                                                                                 \
      meet[tid] = acc;                                                                                                 \
      __syncthreads();                                                                                                 \
      if (tt == 0) {                                                                                                   \
        acc = 0.0;                                                                                                     \
        for (int t = 0; t < TT; ++t) acc += meet[t * RB + lane];                                                       \
      }                                                                                                                \
    }                                                                                                                  \
    if (kFuse) {                                                                                                       \
      /* running arg-max with the generated code's tie rule (replace unless strictly greater); a class */              \
      /* without trees scores the initial value */                                                                     \
      const float m = (float)(s.initialValue + acc);                                                                   \
      if (!(best > m)) { best = m; bestClass = curClass; }                                                             \
      const float m0 = (float)s.initialValue;                                                                          \
      for (int c = curClass + 1; c < (UPTO); ++c)                                                                      \
        if (!(best > m0)) { best = m0; bestClass = c; }                                                                \
    } else if (tt == 0 && lane < valid) {                                                                              \
      partialRow[curClass] = acc;                                                                                      \
      for (int c = curClass + 1; c < (UPTO); ++c) partialRow[c] = 0.0;                                                 \
    }                                                                                                                  \
    acc = 0.0;                                                                                                         \
  }
  // The same where the class is the tree thread's own: nobody to meet.
#define TBAMD_FLUSH_OWN_CLASS(UPTO)                                                                                    \
  {                                                                                                                    \
    if (kFuse) {                                                                                                       \
      const float m = (float)(s.initialValue + acc);                                                                   \
      if (curClass < C && !(best > m)) { best = m; bestClass = curClass; }                                             \
      const float m0 = (float)s.initialValue;                                                                          \
      for (int c = curClass + TT; c < (UPTO); c += TT)                                                                 \
        if (!(best > m0)) { best = m0; bestClass = c; }                                                                \
    } else if (curClass < C && lane < valid) { /* (more tree threads than classes: some have none) */                  \
      partialRow[curClass] = acc;                                                                                      \
      for (int c = curClass + TT; c < (UPTO); c += TT) partialRow[c] = 0.0;                                            \
    }                                                                                                                  \
    acc = 0.0;                                                                                                         \
  }
  // Walks the first 64 (or fewer) entries of the wave's queue to their leaves, one entry per lane, and adds the
  // leaf values to the sums of the rows they belong to; what the queue holds beyond 64 moves to its front.  A
  // lane without an entry walks tail node 0, a leaf of value 0.  Only LDS accesses of this one wave touch the
  // queue, and a wave's LDS accesses complete in program order.
  const uint32_t tileShift = (uint32_t)__builtin_ctz((unsigned)RB) + 2u; // feature index -> byte offset in the row tile
#define TBAMD_WALK_QUEUE                                                                                               \
  {                                                                                                                    \
    const uint32_t me = (uint32_t)(tid & 63);                                                                          \
    const uint32_t take = queued < 64u ? queued : 64u;                                                                 \
    const uint32_t entry = me < take ? queue[me] : 0u;                                                                 \
    const uint32_t later = 64u + me < queued ? queue[64u + me] : 0u;                                                   \
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");                                                             \
    __builtin_amdgcn_wave_barrier();                                                                                   \
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");                                                             \
    handBack[me] = 0.0;                                                                                                \
    uint32_t at = entry & kStubIndexMask;                                                                              \
    const uint32_t owner = entry >> 26;                                                                                \
    const uint32_t ownerColumn = waveColumn + owner * 4u;                                                              \
    U32x2 node = tailNodes[at];                                                                                        \
    for (int d = 0; d < s.tailDepth; ++d) {                                                                            \
      const bool left = LdsLoadFloat(ownerColumn + ((node.y & ((1u << kTailFeatureBits) - 1u)) << tileShift)) < AsFloat(node.x); \
      const uint32_t next = (node.y >> kTailFeatureBits) + (left ? 0u : 1u);                                           \
      const bool moved = next != at;                                                                                   \
      at = next;                                                                                                       \
      if (!__any(moved)) break;                                                                                        \
      node = tailNodes[at];                                                                                            \
    }                                                                                                                  \
    const double leafValue = (double)AsFloat(node.x);                                                                  \
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");                                                             \
    __builtin_amdgcn_wave_barrier();                                                                                   \
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");                                                             \
    if (me < take) __hip_atomic_fetch_add(&handBack[owner], leafValue, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT); \
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");                                                             \
    __builtin_amdgcn_wave_barrier();                                                                                   \
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");                                                             \
    acc += handBack[me];                                                                                               \
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");                                                             \
    __builtin_amdgcn_wave_barrier();                                                                                   \
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");                                                             \
    if (64u + me < queued) queue[me] = later;                                                                          \
    queued = queued > 64u ? queued - 64u : 0u;                                                                         \
  }
  if (PF > 0 && gBegin < gEnd) TBAMD_PREFETCH_GROUP(groups[gBegin])

  for (int g = gBegin; g < gEnd; ++g) {
    const DeviceGroup grp = groups[g];
    if (PF > 0 || g > gBegin) { // rows staged / previous group no longer read
      // (leaf values may still be on their way: only LDS accesses are waited for)
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
    }
    if (PF > 0) {
      U32x4 *dst = reinterpret_cast<U32x4 *>(lds);
      const int pieces = (int)(grp.nodeCount >> 1);
#pragma unroll
      for (int i = 0; i < PF; ++i) {
        const int idx = tid + i * threads;
        if (idx < pieces) dst[idx] = fetched[i];
      }
    } else {
      if (g > gBegin) TBAMD_COPY_GROUP(grp)
      __builtin_amdgcn_s_waitcnt(0x0F70);
      asm volatile("" ::: "memory");
    }
    __syncthreads();
    if (PF > 0 && g + 1 < gEnd) TBAMD_PREFETCH_GROUP(groups[g + 1]) // in flight while this group is walked

    // Walking waves go before waves that are staging (this block's or the other block's on the CU): the walk is
    // what keeps the LDS and the VALUs busy.
    __builtin_amdgcn_s_setprio(1);
    // Bundles are sorted by class; a segment is a run of bundles of one class.
    uint32_t b0 = 0;
    while (b0 < grp.bundleCount) {
      uint32_t b1 = grp.bundleCount;
      if (C > 0 && !own) {
        // most groups vote for one class: the descriptor says so and no bundle has to be looked at
        const int cls = grp.uniformClass ? (int)grp.uniformClass - 1 : (int)bundles[grp.bundleBegin + b0].classId;
        if (cls != curClass) { // classes arrive in ascending order
          TBAMD_ADD_LEAVES
          TBAMD_FLUSH_CLASS(cls)
          curClass = cls;
        }
        if (!grp.uniformClass) {
          b1 = b0 + 1;
          while (b1 < grp.bundleCount && (int)bundles[grp.bundleBegin + b1].classId == cls) ++b1;
        }
      }
      for (uint32_t b = b0 + tt; b < b1; b += TT) {
        // A bundle and its roots are asked for together and awaited once.  (Left to itself the compiler waits for the depth before it
        // asks for the roots, a scalar round trip more a bundle: 2^20 rows x 800 trees x 8 classes 741 -> 727 us, x 1000 trees 1057 -> 1050.
        // Walks with deferred tails have none to gain: 65536 rows x 40 deep trees 24.1 -> 24.4.)
        const DeviceBundle bd = bundles[grp.bundleBegin + b];
        DeviceNode roots[K];
        if (kMode != kTileRankU8) {
#pragma unroll
          for (int k = 0; k < K; ++k) roots[k] = bundleRoots[(size_t)(grp.bundleBegin + b) * K + k];
#pragma unroll
          for (int k = 0; k < K && !kDefer; ++k) asm volatile("" ::"s"(roots[k].meta), "s"(bd.depth));
        }
        if (own && (int)bd.classId != curClass) {
          TBAMD_ADD_LEAVES
          TBAMD_FLUSH_OWN_CLASS((int)bd.classId)
          curClass = (int)bd.classId;
        }
        uint32_t addr[K];
#pragma unroll
        for (int k = 0; k < K; ++k) addr[k] = bd.root[k];
        const int depth = (int)bd.depth;
        // Level 0 of the f32 tiles: copies of the root nodes sit next to the bundles and arrive in scalar
        // registers, only the feature is read from LDS.  A root that is a leaf holds the walk in place like any other leaf, so the step is safe
        // for depth 0.  (On rank tiles, whose rounds are latency-bound, the extra scalar load did not pay.)
        // (the last level's leaves stand 4 bytes apart)
        const uint32_t lastRight = kOutside || (kDump && s.leavesOutside) ? 4u : kNodeBytes;
        const uint32_t rootRight = (kOutside || kDump) && depth == 1 ? lastRight : kNodeBytes;
        if (kMode != kTileRankU8) {
#pragma unroll
          for (int k = 0; k < K; ++k) {
            const DeviceNode root = roots[k];
            const uint32_t off = kMode == kTileF32Words ? MetaFeature(root.meta) << 2 : MetaFeature(root.meta);
            bool left;
            if (kMode == kTileRankU16) left = RankGoesLeft<kMode>(column + off, __float_as_uint(root.value));
            else left = LdsLoadFloat(column + off) < root.value;
            addr[k] = MetaChild(root.meta) + (left ? 0u : rootRight);
          }
        }
        const auto step = [&](uint32_t right) {
#pragma unroll
          for (int k = 0; k < K; ++k) {
            const U32x2 node = LdsLoadNode(addr[k]);
            const uint32_t off = kMode == kTileF32Bytes || kMode == kTileRankU16 ? MetaFeature(node.y) : MetaFeature(node.y) << 2;
            bool left;
            if (IsRankTile(kMode)) left = RankGoesLeft<kMode>(column + off, node.x); // rank <= threshold index
            else left = LdsLoadFloat(column + off) < AsFloat(node.x);
            addr[k] = AddChild(node.y, left ? 0u : right);
          }
        };
        constexpr int kFirstLevel = kMode != kTileRankU8 ? 1 : 0;
#pragma unroll 2
        for (int d = kFirstLevel; d < depth - (kOutside || kDump ? 1 : 0); ++d) step(kNodeBytes);
        if ((kOutside || kDump) && depth > kFirstLevel) step(lastRight);
        if (kDefer && bd.hasStubs) {
          // rows on a stub are queued, the others add their leaf; the queue is walked on as soon as it holds a wave's worth
          float value[K];
#pragma unroll
          for (int k = 0; k < K; ++k) value[k] = LdsLoadFloat(addr[k]);
#pragma unroll
          for (int k = 0; k < K; ++k) {
            const bool stub = __builtin_amdgcn_classf(value[k], 0x3); // a stub's value is a NaN (no leaf's is)
            acc += (double)(stub ? 0.0f : value[k]);
            const uint64_t who = __ballot(stub);
            if (who != 0) {
              const uint32_t before = __builtin_amdgcn_mbcnt_hi((uint32_t)(who >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)who, 0u));
              // entry: the NaN's payload (index of the node the stub stands for) below the lane's number
              if (stub) queue[queued + before] = (__float_as_uint(value[k]) & kStubIndexMask) | laneTag;
              queued += (uint32_t)__builtin_popcountll(who);
              if (queued >= 64u) TBAMD_WALK_QUEUE
            }
          }
        } else {
          if (kDump && s.deferTails && bd.hasStubs) {
            // the dump walks the rows that stand on a stub on at once, each lane for itself, through the tail array
#pragma unroll
            for (int k = 0; k < K; ++k) {
              const float stop = LdsLoadFloat(addr[k]);
              if (__builtin_amdgcn_classf(stop, 0x3)) {
                uint32_t at = __float_as_uint(stop) & kStubIndexMask;
                U32x2 node = tailNodes[at];
                for (int d = 0; d < s.tailDepth; ++d) {
                  const bool left = LdsLoadFloat(column + ((node.y & ((1u << kTailFeatureBits) - 1u)) << tileShift)) < AsFloat(node.x);
                  at = (node.y >> kTailFeatureBits) + (left ? 0u : 1u);
                  node = tailNodes[at];
                }
                acc += (double)AsFloat(node.x);
                const int tree = slotTree[bd.firstSlot + k];
                if (lane < valid && tree >= 0) leafIds[row * s.numTrees + tree] = tailOrigin[at];
                addr[k] = 0; // (the null leaf: adds 0 below and names no tree's node)
              }
            }
          }
          const char *image = reinterpret_cast<const char *>(nodes16) + (size_t)grp.nodeBegin * kNodeBytes;
          TBAMD_ADD_LEAVES
#pragma unroll
          for (int k = 0; k < K; ++k) {
            if (kOutside) leaf[k] = *reinterpret_cast<const float *>(image + addr[k]);
            else if (kDump) acc += (double)*reinterpret_cast<const float *>(image + addr[k]);
            else acc += (double)LdsLoadFloat(addr[k]);
          }
        }
        if (kDump) {
          if (lane < valid) {
#pragma unroll
            for (int k = 0; k < K; ++k) {
              const int tree = slotTree[bd.firstSlot + k];
              if (tree >= 0 && !(s.deferTails && addr[k] == 0u))
                leafIds[row * s.numTrees + tree] = nodeOrigin[grp.nodeBegin * 2u + addr[k] / 4u];
            }
          }
        }
      }
      b0 = b1;
    }
    __builtin_amdgcn_s_setprio(0);
  }
  if (kDefer) // what is still queued is walked on now
    while (queued > 0u) TBAMD_WALK_QUEUE

  TBAMD_ADD_LEAVES
  if (own) {
    TBAMD_FLUSH_OWN_CLASS(C)
    if (!kFuse) return;
    // each tree thread has the best of its own classes: the larger sum, or the larger class id of equal ones, as the running rule
    // (and of sums that are no numbers, by a base score that is none; a thread without a class has -inf and class 0)
    __syncthreads();
    float *bests = reinterpret_cast<float *>(lds);
    int *classes = reinterpret_cast<int *>(lds) + threads;
    bests[tid] = best;
    classes[tid] = bestClass;
    __syncthreads();
    if (tt != 0 || lane >= valid) return;
    for (int t = 1; t < TT; ++t) {
      const float m = bests[t * RB + lane];
      const int c = classes[t * RB + lane];
      if (m > best || (!(best > m) && c > bestClass)) { best = m; bestClass = c; }
    }
    if (classOut) classOut[row] = (int8_t)bestClass;
    else out[row] = (float)bestClass;
    return;
  }
  if (C > 0) {
    TBAMD_FLUSH_CLASS(C)
    if (kFuse && tt == 0 && lane < valid) {
      if (classOut) classOut[row] = (int8_t)bestClass;
      else out[row] = (float)bestClass;
    }
    return;
  }
  if (TT > 1) {
    __syncthreads();
    meet[tid] = acc;
    __syncthreads();
    if (tt != 0) return;
    acc = 0.0;
    for (int t = 0; t < TT; ++t) acc += meet[t * RB + lane];
  }
  if (lane >= valid) return;
  if (partial) {
    partialRow[0] = acc;
  } else {
    const double margin = s.initialValue + acc;
    out[row] = (float)(s.transform == 1 ? 1.0 / (1.0 + exp(-margin)) : margin);
  }
#undef TBAMD_COPY_GROUP
#undef TBAMD_ADD_LEAVES
#undef TBAMD_FLUSH_CLASS
#undef TBAMD_FLUSH_OWN_CLASS
#undef TBAMD_PREFETCH_GROUP
#undef TBAMD_WALK_QUEUE
}

template <int K, int PF, int kMode, int kVariant>
__global__ void __launch_bounds__(1024)
WalkRowsLdsKernel(const float *__restrict__ x, const uint4 *__restrict__ nodes16,
                  const DeviceBundle *__restrict__ bundles, const DeviceNode *__restrict__ bundleRoots,
                  const DeviceGroup *__restrict__ groups,
                  const WalkScalars s, float *__restrict__ out, int8_t *__restrict__ classOut,
                  double *__restrict__ partial, int32_t *__restrict__ leafIds, const int32_t *__restrict__ nodeOrigin,
                  const int32_t *__restrict__ slotTree, const U32x2 *__restrict__ tailNodes, const int32_t *__restrict__ tailOrigin) {
  extern __shared__ __align__(16) unsigned char lds[];
  const int slice = blockIdx.y;
  const int gBegin = (int)(((int64_t)s.numGroups * slice) / s.treeSlices);
  const int gEnd = (int)(((int64_t)s.numGroups * (slice + 1)) / s.treeSlices);
  WalkRowBlock<K, PF, kMode, kVariant>(lds, blockIdx.x, gBegin, gEnd, slice, x, nodes16, bundles, bundleRoots, groups, s, out, classOut,
                                       partial, leafIds, nodeOrigin, slotTree, tailNodes, tailOrigin);
}

// ---------------------------------------------------------------------------
// The row-parallel walk for batches of a few rounds of blocks.  Row blocks x tree groups are one line of units, cut
// into as many equal parts as blocks run at once: no last round that is nearly empty (65537 rows in blocks of 256 x 2
// tree slices are 514 blocks for 512 places, which took twice the time of 512), and a block stages the rows of the row
// blocks its part touches, one or two.  Part p of a row block leaves its sums in slot p of the partial sums, which the
// finalize kernel adds in order.  (Adding them in the block that comes last, found with a ticket, was measured: the
// write-through stores, the ticket and the reads are three round trips to memory, 5 to 12 us where the finalize launch
// takes 4.)
// ---------------------------------------------------------------------------
template <int K, int kMode, int kVariant> // kWalkPlain or kWalkOwn, their leaves in LDS or not
// (80 SGPRs: with the 16 the trap handler takes, 8 waves per SIMD - two blocks of 16 waves - leave each wave 100; at 88 one
// block per CU ran, 40 % slower)
__global__ void __launch_bounds__(1024) __attribute__((amdgpu_num_sgpr(80)))
WalkRowsSplitKernel(const float *__restrict__ x, const uint4 *__restrict__ nodes16,
                    const DeviceBundle *__restrict__ bundles, const DeviceNode *__restrict__ bundleRoots,
                    const DeviceGroup *__restrict__ groups, const WalkScalars s, double *__restrict__ partial) {
  extern __shared__ __align__(16) unsigned char lds[];
  const SplitLine line{((s.rows + s.rowsPerBlock - 1) / s.rowsPerBlock) * s.numGroups, s.numGroups, (int)gridDim.x};
  WalkScalars own = s;
  int64_t unit = line.FirstUnit(blockIdx.x);
  const int64_t unitEnd = line.FirstUnit((int64_t)blockIdx.x + 1);
  while (unit < unitEnd) {
    // (what the walk computes from these is computed again for every row block, not kept in registers across them)
    asm volatile("" : "+s"(own.rowsPerBlock), "+s"(own.numFeatures), "+s"(own.treeThreads), "+s"(own.groupRegionBytes));
    const int64_t rowBlock = unit / line.groups;
    const int gBegin = (int)(unit - rowBlock * line.groups);
    const int64_t left = unitEnd - rowBlock * line.groups;
    const int gEnd = (int)(left < line.groups ? left : line.groups);
    WalkRowBlock<K, 0, kMode, kVariant>(lds, rowBlock, gBegin, gEnd, (int)((int64_t)blockIdx.x - line.FirstBlock(rowBlock)), x, nodes16,
                                          bundles, bundleRoots, groups, own, nullptr, nullptr, partial, nullptr, nullptr, nullptr, nullptr,
                                          nullptr);
    unit += gEnd - gBegin;
    __syncthreads(); // the rows' tile and the group are rewritten
  }
}

// ---------------------------------------------------------------------------
// Row-parallel walk over TILED trees (tiles of T = 2 to 8 nodes, layout in device_model.h): the
// reference's tile step (src/mlir/CodeGenStateMachine.cpp:284-506, cooperative GPU form
// src/gpu/GPUSimtPass.cpp:39-133) as branch-free per-lane code.  One step reads the tile (thresholds,
// feature offsets, child base and the tile's own child-select row) with one to four wide LDS reads, gathers
// the T feature values of the lane's row, turns the T comparisons into an outcome word (node i in bit i)
// and picks the child out of the select row with one shift (tiles of up to 4 nodes) or by following the
// tile's links (the eight-slot tile of tile sizes 5 to 8).  Leaves are tiles that select themselves, so a
// bundle walks `depth` tile steps without a leaf test.  Block shape, row tile, tree groups (staged by direct
// global-to-LDS copies), tree threads, class flush and epilogue are those of WalkRowsLdsKernel.
//
// Bundles carry a peel depth (taken from a hit-count profile: the steps that bring 90 % of the profiled
// rows to a leaf, src/mlir/ProbabilityBasedTilingTransform.cpp:66-73; equal to the depth without one): the
// walk takes that many steps blind and then goes on only while some lane of the wave still moves, at most to
// the full depth.
// ---------------------------------------------------------------------------
typedef const __attribute__((address_space(3))) U32x4 *LdsQuadPtr;
__device__ __forceinline__ U32x4 LdsLoadQuad(uint32_t address) { return *(LdsQuadPtr)(uintptr_t)address; }

template <int T> // 2, 3, 4, or kMaxTileSize for the eight-slot tile of tile sizes 5 to 8
__device__ __forceinline__ uint32_t TileStep(uint32_t addr, uint32_t column, int hops) {
  static_assert(T >= 2 && (T <= kMaxSelectTile || T == kMaxTileSize), "tile sizes 5 to 8 share the eight-slot tile");
  float thr[T];
  uint32_t off[T];
  uint32_t childBase;
  uint64_t select; // the child-select row, or the links of the eight-slot tile
  if constexpr (T == 2) {
    const U32x4 q = LdsLoadQuad(addr);
    thr[0] = AsFloat(q.x), thr[1] = AsFloat(q.y);
    off[0] = q.z & 0xFFFFu, off[1] = q.z >> 16;
    childBase = q.w & 0xFFFFu;
    select = q.w >> 16;
  } else if constexpr (T == 3) {
    const U32x2 a = LdsLoadNode(addr), b = LdsLoadNode(addr + 8), c = LdsLoadNode(addr + 16);
    thr[0] = AsFloat(a.x), thr[1] = AsFloat(a.y), thr[2] = AsFloat(b.x);
    off[0] = b.y & 0xFFFFu, off[1] = b.y >> 16, off[2] = c.x & 0xFFFFu;
    childBase = c.x >> 16;
    select = c.y & 0xFFFFu;
  } else if constexpr (T == 4) {
    const U32x4 q0 = LdsLoadQuad(addr), q1 = LdsLoadQuad(addr + 16);
    thr[0] = AsFloat(q0.x), thr[1] = AsFloat(q0.y), thr[2] = AsFloat(q0.z), thr[3] = AsFloat(q0.w);
    off[0] = q1.x & 0xFFFFu, off[1] = q1.x >> 16, off[2] = q1.y & 0xFFFFu, off[3] = q1.y >> 16;
    childBase = q1.z & 0xFFFFu;
    select = (uint64_t)(q1.z >> 16) | ((uint64_t)q1.w << 16);
  } else {
    const U32x4 q0 = LdsLoadQuad(addr), q1 = LdsLoadQuad(addr + 16), q2 = LdsLoadQuad(addr + 32), q3 = LdsLoadQuad(addr + 48);
    thr[0] = AsFloat(q0.x), thr[1] = AsFloat(q0.y), thr[2] = AsFloat(q0.z), thr[3] = AsFloat(q0.w);
    thr[4] = AsFloat(q1.x), thr[5] = AsFloat(q1.y), thr[6] = AsFloat(q1.z), thr[7] = AsFloat(q1.w);
    off[0] = q2.x & 0xFFFFu, off[1] = q2.x >> 16, off[2] = q2.y & 0xFFFFu, off[3] = q2.y >> 16;
    off[4] = q2.z & 0xFFFFu, off[5] = q2.z >> 16, off[6] = q2.w & 0xFFFFu, off[7] = q2.w >> 16;
    select = (uint64_t)q3.x | ((uint64_t)q3.y << 32);
    childBase = q3.z & 0xFFFFu;
  }
  if constexpr (T > kMaxSelectTile) {
    // The eight comparisons pick, slot by slot, the link the slot sends its row along: nibble s of the high word
    // of `select` when slot s sends the row left, nibble s of the low word otherwise (one bit-field insert under a
    // mask of eight nibbles).  Then the links are followed from slot 0: a link below kTileLinkExit names the next
    // slot (link + 1), the others the child; a tile holds `hops` levels of nodes, so `hops` links reach a child.
    uint32_t wentLeft = 0;
#pragma unroll
    for (int i = 0; i < T; ++i) {
      const float x = LdsLoadFloat(column + off[i]);
      wentLeft |= x < thr[i] ? 0xFu << (4 * i) : 0u;
    }
    const uint32_t taken = ((uint32_t)(select >> 32) & wentLeft) | ((uint32_t)select & ~wentLeft);
    uint32_t link = taken & 15u;
    for (int hop = 1; hop < hops; ++hop) {
      const uint32_t next = __builtin_amdgcn_ubfe(taken, (link + 1u) << 2, 4u); // (the field offset wraps at 32 for a link that names a child: ignored below)
      link = link < kTileLinkExit ? next : link;
    }
    return childBase + (link - kTileLinkExit) * TileBytes(T);
  } else {
    uint32_t outcome = 0;
#pragma unroll
    for (int i = 0; i < T; ++i) {
      const float x = LdsLoadFloat(column + off[i]);
      outcome |= (x < thr[i] ? 1u : 0u) << i;
    }
    const uint32_t child = (uint32_t)(select >> (outcome * TileSelectBits(T))) & ((1u << TileSelectBits(T)) - 1u);
    return childBase + child * TileBytes(T);
  }
}

template <int T, int K, int kVariant> // kVariant: kWalkPlain, kWalkDump or kWalkFuse (the peel tail is always there)
__global__ void __launch_bounds__(1024)
WalkRowsTiledKernel(const float *__restrict__ x, const uint4 *__restrict__ nodes16,
                    const DeviceBundle *__restrict__ bundles, const DeviceGroup *__restrict__ groups,
                    const WalkScalars s, float *__restrict__ out, int8_t *__restrict__ classOut,
                    double *__restrict__ partial, int32_t *__restrict__ leafIds, const int32_t *__restrict__ nodeOrigin,
                    const int32_t *__restrict__ slotTree) {
  constexpr bool kDump = kVariant == kWalkDump, kFuse = kVariant == kWalkFuse;
  extern __shared__ __align__(16) unsigned char lds[];
  const int tid = threadIdx.x;
  const int threads = blockDim.x;
  const int RB = s.rowsPerBlock;
  const int TT = s.treeThreads;
  const int lane = tid & (RB - 1);
  const int tt = __builtin_amdgcn_readfirstlane(tid / RB);
  const int F = s.numFeatures;
  const int64_t row0 = (int64_t)blockIdx.x * RB;
  const int64_t remaining = s.rows - row0;
  const int valid = remaining < RB ? (int)remaining : RB;

  float *rowTile = reinterpret_cast<float *>(lds + s.groupRegionBytes);
  StageRowsTransposed(x + row0 * F, valid, RB, F, rowTile, tid, threads);
  for (int i = tid; i < RB; i += threads) rowTile[F * RB + i] = -INFINITY; // pad feature: keeps leaves in place
  const uint32_t column = s.groupRegionBytes + (uint32_t)lane * 4u;

  const int slice = blockIdx.y;
  const int gBegin = (int)(((int64_t)s.numGroups * slice) / s.treeSlices);
  const int gEnd = (int)(((int64_t)s.numGroups * (slice + 1)) / s.treeSlices);
  const int C = s.numClasses;
  const int64_t row = row0 + lane;
  double *partialRow = partial ? partial + ((int64_t)slice * s.rows + row) * (C > 0 ? C : 1) : nullptr;
  double *meet = reinterpret_cast<double *>(C > 0 ? lds + ((s.groupRegionBytes + (uint32_t)(F + 1) * RB * 4u + 7u) & ~7u) : lds);

  double acc = 0.0;
  int curClass = 0;
  float best = -INFINITY; // fuseArgmax: running maximum of the class sums and its class (tree thread 0)
  int bestClass = 0;
#define TBAMD_FLUSH_CLASS(UPTO)                                                                                        \
  {                                                                                                                    \
    if (TT > 1) {                                                                                                      \
      __syncthreads();                                                                                                 \
      meet[tid] = acc;                                                                                                 \
      __syncthreads();                                                                                                 \
      if (tt == 0) {                                                                                                   \
        acc = 0.0;                                                                                                     \
        for (int t = 0; t < TT; ++t) acc += meet[t * RB + lane];                                                       \
      }                                                                                                                \
    }                                                                                                                  \
    if (kFuse) {                                                                                                \
      /* running arg-max with the generated code's tie rule (replace unless strictly greater); a class */              \
      /* without trees scores the initial value */                                                                     \
      const float m = (float)(s.initialValue + acc);                                                                   \
      if (!(best > m)) { best = m; bestClass = curClass; }                                                             \
      const float m0 = (float)s.initialValue;                                                                          \
      for (int c = curClass + 1; c < (UPTO); ++c)                                                                      \
        if (!(best > m0)) { best = m0; bestClass = c; }                                                                \
    } else if (tt == 0 && lane < valid) {                                                                              \
      partialRow[curClass] = acc;                                                                                      \
      for (int c = curClass + 1; c < (UPTO); ++c) partialRow[c] = 0.0;                                                 \
    }                                                                                                                  \
    acc = 0.0;                                                                                                         \
  }
  for (int g = gBegin; g < gEnd; ++g) {
    const DeviceGroup grp = groups[g];
    __syncthreads();
    {
      // The group goes straight from global memory into LDS (lane i of a wave-wide load leaves its 16 bytes at
      // base + 16 i, lanes switched off write nothing), as in the scalar kernel's direct form.
      const U32x4 *src = reinterpret_cast<const U32x4 *>(nodes16) + (grp.nodeBegin >> 1);
      const int pieces = (int)(grp.nodeCount >> 1);
      const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
      for (int first = wave * 64; first < pieces; first += threads)
        if (first + (tid & 63) < pieces)
          __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)(src + first + (tid & 63)),
                                           (__attribute__((address_space(3))) void *)(lds + (uint32_t)first * 16u), 16, 0, 0);
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
    __syncthreads();

    uint32_t b0 = 0;
    while (b0 < grp.bundleCount) {
      uint32_t b1 = grp.bundleCount;
      if (C > 0) {
        const int cls = grp.uniformClass ? (int)grp.uniformClass - 1 : (int)bundles[grp.bundleBegin + b0].classId;
        if (cls != curClass) {
          TBAMD_FLUSH_CLASS(cls)
          curClass = cls;
        }
        if (!grp.uniformClass) {
          b1 = b0 + 1;
          while (b1 < grp.bundleCount && (int)bundles[grp.bundleBegin + b1].classId == cls) ++b1;
        }
      }
      for (uint32_t b = b0 + tt; b < b1; b += TT) {
        const DeviceBundle bd = bundles[grp.bundleBegin + b];
        uint32_t addr[K];
#pragma unroll
        for (int k = 0; k < K; ++k) addr[k] = bd.root[k];
        const int depth = (int)bd.depth;
        const int blind = (int)bd.peelDepth;
        for (int d = 0; d < blind; ++d) {
#pragma unroll
          for (int k = 0; k < K; ++k) addr[k] = TileStep<T>(addr[k], column, s.tileHops);
        }
        for (int d = blind; d < depth; ++d) {
          bool moved = false;
#pragma unroll
          for (int k = 0; k < K; ++k) {
            const uint32_t next = TileStep<T>(addr[k], column, s.tileHops);
            moved = moved || next != addr[k];
            addr[k] = next;
          }
          if (!__any(moved)) break; // every lane of the wave sits on a leaf tile (leaves select themselves)
        }
#pragma unroll
        for (int k = 0; k < K; ++k) acc += (double)LdsLoadFloat(addr[k]);
        if (kDump) {
          if (lane < valid) {
#pragma unroll
            for (int k = 0; k < K; ++k) {
              const int tree = slotTree[bd.firstSlot + k];
              if (tree >= 0) leafIds[row * s.numTrees + tree] = nodeOrigin[grp.nodeBegin * 2u + addr[k] / 4u];
            }
          }
        }
      }
      b0 = b1;
    }
  }

  if (C > 0) {
    TBAMD_FLUSH_CLASS(C)
    if (kFuse && tt == 0 && lane < valid) {
      if (classOut) classOut[row] = (int8_t)bestClass;
      else out[row] = (float)bestClass;
    }
    return;
  }
  if (TT > 1) {
    __syncthreads();
    meet[tid] = acc;
    __syncthreads();
    if (tt != 0) return;
    acc = 0.0;
    for (int t = 0; t < TT; ++t) acc += meet[t * RB + lane];
  }
  if (lane >= valid) return;
  if (partial) {
    partialRow[0] = acc;
  } else {
    const double margin = s.initialValue + acc;
    out[row] = (float)(s.transform == 1 ? 1.0 / (1.0 + exp(-margin)) : margin);
  }
#undef TBAMD_FLUSH_CLASS
}

// ---------------------------------------------------------------------------
// Tree-parallel walk.  The block keeps `rowsPerBlock` rows row-major in LDS and
// gives each row `treeLanes` lanes; lane j of a row walks bundles j, j+treeLanes,
// ... of the staged tree group, so a row's trees are shared between its lanes.
// The lanes' partial sums are combined with a wave-level butterfly (lanes of a
// row are contiguous), then across waves through LDS when a row spans several
// waves.  One lane per row owns the row's per-class accumulators in LDS, which
// keeps the summation order fixed.  Used when a row is too wide to transpose
// 64 of them into LDS, and when the batch has too few rows to fill the chip
// with one lane per row.
// ---------------------------------------------------------------------------
// One butterfly step on doubles.  Partners 1, 2, 4 and 8 lanes away are reached with DPP operand swizzles
// inside the VALU (quad permutes, the mirror of half a row and of a row: after the steps before them every
// lane of the mirrored group already holds the same partial sum, so the mirror partner is as good as the
// xor partner); only the steps across rows of 16 lanes go through the LDS crossbar (ds_bpermute).
template <int kDppCtrl>
__device__ __forceinline__ double DppMove(double v) {
  int lo = __double2loint(v), hi = __double2hiint(v);
  lo = __builtin_amdgcn_update_dpp(0, lo, kDppCtrl, 0xF, 0xF, false);
  hi = __builtin_amdgcn_update_dpp(0, hi, kDppCtrl, 0xF, 0xF, false);
  return __hiloint2double(hi, lo);
}

__device__ __forceinline__ double ShuffleXor(double v, int mask) {
  switch (mask) {
  case 1: return DppMove<0xB1>(v);  // quad_perm [1,0,3,2]
  case 2: return DppMove<0x4E>(v);  // quad_perm [2,3,0,1]
  case 4: return DppMove<0x141>(v); // row_half_mirror
  case 8: return DppMove<0x140>(v); // row_mirror
  default: break;
  }
  int lo = __double2loint(v), hi = __double2hiint(v);
  lo = __shfl_xor(lo, mask, 64);
  hi = __shfl_xor(hi, mask, 64);
  return __hiloint2double(hi, lo);
}

template <int K, int PF, bool kDump>
__global__ void __launch_bounds__(1024)
WalkTreeParallelKernel(const float *__restrict__ x, const uint4 *__restrict__ nodes16,
                       const DeviceBundle *__restrict__ bundles, const DeviceGroup *__restrict__ groups,
                       const WalkScalars s, float *__restrict__ out, double *__restrict__ partial,
                       int32_t *__restrict__ leafIds, const int32_t *__restrict__ nodeOrigin,
                       const int32_t *__restrict__ slotTree) {
  // LDS: [tree group nodes | rows, (F+1) floats each | cross-wave scratch | per-row class sums]
  extern __shared__ __align__(16) unsigned char lds[];
  const int tid = threadIdx.x;
  const int threads = blockDim.x;
  const int F = s.numFeatures;
  const int R = s.rowsPerBlock;
  const int TL = s.treeLanes;
  const int r = tid / TL;
  const int j = tid - r * TL;
  const int C = s.numClasses;
  const int Cn = C > 0 ? C : 1;
  const int64_t row0 = (int64_t)blockIdx.x * R;
  const int64_t remaining = s.rows - row0;
  const int valid = remaining < R ? (int)remaining : R;
  const int rowWords = F + 1;

  float *rowsLds = reinterpret_cast<float *>(lds + s.groupRegionBytes);
  const uint32_t scratchOffset = (s.groupRegionBytes + (uint32_t)R * rowWords * 4u + 7u) & ~7u;
  double *waveScratch = reinterpret_cast<double *>(lds + scratchOffset);
  double *classSums = waveScratch + (threads + 63) / 64;

  StageRows(x + row0 * F, valid, R, F, rowWords, rowsLds, tid, threads);
  for (int rr = tid; rr < R; rr += threads) rowsLds[rr * rowWords + F] = -INFINITY;
  for (int i = tid; i < R * Cn; i += threads) classSums[i] = 0.0;
  const uint32_t rowBase = s.groupRegionBytes + (uint32_t)r * rowWords * 4u;

  const int slice = blockIdx.y;
  const int gBegin = (int)(((int64_t)s.numGroups * slice) / s.treeSlices);
  const int gEnd = (int)(((int64_t)s.numGroups * (slice + 1)) / s.treeSlices);
  const int64_t row = row0 + r;

  // Register double buffer for the next tree group (loads stay in flight across the walk).
  U32x4 fetched[PF];
#define TBAMD_PREFETCH_GROUP(NEXTGRP)                                                                                  \
  {                                                                                                                    \
    const DeviceGroup nextGrp = (NEXTGRP);                                                                             \
    const U32x4 *src = reinterpret_cast<const U32x4 *>(nodes16) + (nextGrp.nodeBegin >> 1);                            \
    const int last = (int)(nextGrp.nodeCount >> 1) - 1;                                                                \
    _Pragma("unroll") for (int i = 0; i < PF; ++i) {                                                                   \
      const int idx = tid + i * threads;                                                                               \
      fetched[i] = src[idx < last ? idx : last];                                                                       \
    }                                                                                                                  \
  }
  if (gBegin < gEnd) TBAMD_PREFETCH_GROUP(groups[gBegin])

  for (int g = gBegin; g < gEnd; ++g) {
    const DeviceGroup grp = groups[g];
    __syncthreads();
    {
      U32x4 *dst = reinterpret_cast<U32x4 *>(lds);
      const int pieces = (int)(grp.nodeCount >> 1);
#pragma unroll
      for (int i = 0; i < PF; ++i) {
        const int idx = tid + i * threads;
        if (idx < pieces) dst[idx] = fetched[i];
      }
    }
    __syncthreads();
    if (g + 1 < gEnd) TBAMD_PREFETCH_GROUP(groups[g + 1])

    // bundles are sorted by class: handle one class segment at a time
    uint32_t b0 = 0;
    while (b0 < grp.bundleCount) {
      const int cls = bundles[grp.bundleBegin + b0].classId;
      uint32_t b1 = b0 + 1;
      while (b1 < grp.bundleCount && bundles[grp.bundleBegin + b1].classId == cls) ++b1;

      double acc = 0.0;
      for (uint32_t b = b0 + j; b < b1; b += TL) {
        const DeviceBundle bd = bundles[grp.bundleBegin + b];
        uint32_t addr[K];
#pragma unroll
        for (int k = 0; k < K; ++k) addr[k] = bd.root[k];
        const int depth = bd.depth;
        for (int d = 0; d < depth; ++d) {
#pragma unroll
          for (int k = 0; k < K; ++k) {
            const U32x2 node = LdsLoadNode(addr[k]);
            const float xv = LdsLoadFloat(rowBase + MetaFeature(node.y));
            addr[k] = AddChild(node.y, xv < AsFloat(node.x) ? 0u : kNodeBytes);
          }
        }
#pragma unroll
        for (int k = 0; k < K; ++k) acc += (double)LdsLoadFloat(addr[k]);
        if (kDump) {
          if (r < valid) {
#pragma unroll
            for (int k = 0; k < K; ++k) {
              const int tree = slotTree[bd.firstSlot + k];
              if (tree >= 0) leafIds[row * s.numTrees + tree] = nodeOrigin[grp.nodeBegin * 2u + addr[k] / 4u];
            }
          }
        }
      }

      // combine the lanes of each row: butterfly inside the wave ...
      const int inWave = TL < 64 ? TL : 64;
      for (int m = 1; m < inWave; m <<= 1) acc += ShuffleXor(acc, m); // (ascending: see ShuffleXor)
      if (TL > 64) { // ... then across the row's waves through LDS
        __syncthreads();
        if ((tid & 63) == 0) waveScratch[tid >> 6] = acc;
        __syncthreads();
        if (j == 0) {
          acc = 0.0;
          for (int w = 0; w < TL / 64; ++w) acc += waveScratch[(tid >> 6) + w];
        }
      }
      if (j == 0) classSums[r * Cn + cls] += acc;
      b0 = b1;
    }
  }

  if (j != 0 || r >= valid) return;
  if (C > 0 || partial) {
    double *dst = partial + ((int64_t)slice * s.rows + row) * Cn;
    for (int c = 0; c < Cn; ++c) dst[c] = classSums[r * Cn + c];
  } else {
    const double margin = s.initialValue + classSums[r];
    out[row] = (float)(s.transform == 1 ? 1.0 / (1.0 + exp(-margin)) : margin);
  }
#undef TBAMD_PREFETCH_GROUP
}

// ---------------------------------------------------------------------------
// Global-memory walk: the fallback for forests with a tree that does not fit one LDS group.  One
// lane per row; nodes (16 bytes, absolute child indices) and row values are read from global memory
// through L1/L2, K trees at a time in lock step with an explicit leaf test.  Same accumulation,
// class flush and tree-slice scheme as the LDS kernels.  65536 rows x 28 features, 40 trees of depth 16: 88 us, the texture
// addressers 67 % busy with two gathers a level (node and value), the VALUs 12 %; the rest is the chain of dependent loads.
// ---------------------------------------------------------------------------
template <int K, bool kDump>
__global__ void __launch_bounds__(1024)
WalkGlobalKernel(const float *__restrict__ x, const DeviceGlobalNode *__restrict__ nodes,
                 const DeviceGlobalTree *__restrict__ trees, const WalkScalars s, float *__restrict__ out,
                 double *__restrict__ partial, int32_t *__restrict__ leafIds) {
  const int64_t row = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const bool valid = row < s.rows;
  const float *xr = x + (valid ? row : s.rows - 1) * s.numFeatures;
  const int slice = blockIdx.y;
  const int tBegin = (int)(((int64_t)s.numTrees * slice) / s.treeSlices);
  const int tEnd = (int)(((int64_t)s.numTrees * (slice + 1)) / s.treeSlices);
  const int C = s.numClasses;
  double *partialRow = partial ? partial + ((int64_t)slice * s.rows + (valid ? row : 0)) * (C > 0 ? C : 1) : nullptr;
  typedef uint32_t Quad __attribute__((ext_vector_type(4)));
  const Quad *nodeQuads = reinterpret_cast<const Quad *>(nodes);

  double acc = 0.0;
  int curClass = 0;
  for (int t0 = tBegin; t0 < tEnd; t0 += K) {
    uint32_t n[K];
    uint32_t depth = 0;
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const int t = t0 + k < tEnd ? t0 + k : tEnd - 1; // the tail repeats the last tree; its result is dropped
      n[k] = trees[t].root;
      depth = trees[t].depth > depth ? trees[t].depth : depth;
    }
    for (uint32_t d = 0; d < depth; ++d) {
#pragma unroll
      for (int k = 0; k < K; ++k) {
        const Quad node = nodeQuads[n[k]];
        if (node.y != kGlobalLeaf) n[k] = node.z + (xr[node.y] < AsFloat(node.x) ? 0u : 1u);
      }
    }
#pragma unroll
    for (int k = 0; k < K; ++k) {
      if (t0 + k >= tEnd) break;
      const DeviceGlobalTree tree = trees[t0 + k];
      const Quad leaf = nodeQuads[n[k]];
      if (C > 0 && (int)tree.classId != curClass) { // classes arrive in ascending order
        if (valid) {
          partialRow[curClass] = acc;
          for (int c = curClass + 1; c < (int)tree.classId; ++c) partialRow[c] = 0.0;
        }
        acc = 0.0;
        curClass = (int)tree.classId;
      }
      acc += (double)AsFloat(leaf.x);
      if (kDump && valid) leafIds[row * s.numTrees + tree.origin] = (int32_t)leaf.w;
    }
  }
  if (!valid) return;
  if (C > 0) {
    partialRow[curClass] = acc;
    for (int c = curClass + 1; c < C; ++c) partialRow[c] = 0.0;
  } else if (partial) {
    partialRow[0] = acc;
  } else {
    const double margin = s.initialValue + acc;
    out[row] = (float)(s.transform == 1 ? 1.0 / (1.0 + exp(-margin)) : margin);
  }
}

// ---------------------------------------------------------------------------
// Rank quantisation of the rows.  For every (row, feature) the kernel counts how many of the
// feature's sorted distinct split thresholds are <= the value and writes the count as one byte into
// the tile layout the row-parallel kernel copies verbatim: [block of 64 rows][feature][row].  The
// table is padded with +inf up to 2^n - 1 entries; NaN and +inf count all of them (the largest rank,
// above every node's threshold index, so they go right at every node like the f32 compare sends
// them).  Rows past the end of the batch in the last block get the ranks of the last row; the walk
// never stores their results.
//
// A block owns a chunk of 64 features, whose threshold table sits in LDS as [k][feature]; its waves
// take 64-row blocks in turn.  A lane owns ONE feature of the chunk: whatever level of the search a
// lane is at, lane i reads bank i, so the table reads never conflict, and a wave's row load is 256
// contiguous bytes.  The lane's 64 result bytes pass through a per-wave LDS area (80-byte lane
// stride: conflict-free 16-byte writes) so that the wave stores its 4 KB of tile in four contiguous
// 1 KB pieces.
// ---------------------------------------------------------------------------
constexpr int kBinRows = 64;        // rows per tile = rows per block of the quantised walk
constexpr int kBinFeatures = 64;    // features per block = lanes per wave
constexpr int kBinRowsPerPass = 16; // rows a lane searches side by side
constexpr int kBinWaves = 8;
constexpr int kBinLaneStride = 80;  // bytes of staging per lane (64 used)

// Sixteen rows of one feature, all loads in flight; rows past the batch re-read the last row.
__device__ __forceinline__ void BinLoadRows(const float *__restrict__ x, int64_t rows, int F, int feature, int64_t rowBase,
                                            float (&v)[kBinRowsPerPass]) {
#pragma unroll
  for (int u = 0; u < kBinRowsPerPass; ++u) {
    const int64_t row = rowBase + u;
    v[u] = x[(row < rows ? row : rows - 1) * F + feature];
  }
}

// Ranks of sixteen values of the lane's feature, left as one 16-byte piece at LDS address `piece`.
// Branch-free binary search on byte offsets into the [k][feature] table (lane offset included); every
// level first issues the reads of all rows, then consumes them, so a wave keeps 16 LDS reads in flight.
template <int kLevels>
__device__ __forceinline__ void BinSearchRows(const float (&v)[kBinRowsPerPass], uint32_t laneBytes, unsigned char *piece) {
  typedef uint32_t Piece __attribute__((ext_vector_type(4)));
  constexpr uint32_t strideBytes = kBinFeatures * 4u; // one table level
  uint32_t pos[kBinRowsPerPass];
#pragma unroll
  for (int u = 0; u < kBinRowsPerPass; ++u) pos[u] = laneBytes;
#pragma unroll
  for (int level = kLevels - 1; level >= 0; --level) {
    const uint32_t step = strideBytes << level;
    float probe[kBinRowsPerPass];
#pragma unroll
    for (int u = 0; u < kBinRowsPerPass; ++u) probe[u] = LdsLoadFloat(pos[u] + (step - strideBytes));
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < kBinRowsPerPass; ++u) pos[u] += !(v[u] < probe[u]) ? step : 0u; // NaN: every step taken
    __builtin_amdgcn_sched_barrier(0);
  }
  // byte 1 of every offset is the rank (offset = rank * 256 + lane * 4): gather four of them per word
  uint32_t packed[kBinRowsPerPass / 4];
#pragma unroll
  for (int i = 0; i < kBinRowsPerPass / 4; ++i) {
    const uint32_t lo = __builtin_amdgcn_perm(pos[4 * i + 1], pos[4 * i], 0x0c0c0501u);
    const uint32_t hi = __builtin_amdgcn_perm(pos[4 * i + 3], pos[4 * i + 2], 0x0c0c0501u);
    packed[i] = __builtin_amdgcn_perm(hi, lo, 0x05040100u);
  }
  *reinterpret_cast<Piece *>(piece) = Piece{packed[0], packed[1], packed[2], packed[3]};
}

template <int kLevels> // search depth: the table holds 2^kLevels - 1 thresholds per feature
__global__ void __launch_bounds__(kBinWaves * 64)
BinRowsKernel(const float *__restrict__ x, const float *__restrict__ table, uint8_t *__restrict__ ranks,
              int64_t rows, int F, int rowBlocksPerBlock, int chunks) {
  extern __shared__ __align__(16) unsigned char lds[];
  typedef uint32_t Piece __attribute__((ext_vector_type(4)));
  static_assert(kBinRows == 4 * kBinRowsPerPass, "four passes per row block");
  // Workgroups go to the 8 XCDs in turn, each with its own L2.  A row is not aligned to cache lines
  // (F * 4 bytes is no multiple of 128 in general), so neighbouring feature chunks of the same rows
  // share lines: blocks 8 apart in launch order (same XCD, back to back) take neighbouring chunks of
  // one group of row blocks, and the shared lines are fetched from HBM once.
  const uint32_t linear = blockIdx.x;
  const int chunk = (int)((linear >> 3) % (uint32_t)chunks);
  const int64_t rowGroup = (int64_t)(linear & 7u) + 8 * (int64_t)(linear / (8u * (uint32_t)chunks));
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int f0 = chunk * kBinFeatures;
  const int f = f0 + lane;
  constexpr int depth = (1 << kLevels) - 1;
  constexpr uint32_t tableBytes = (uint32_t)depth * kBinFeatures * 4u;
  {
    float *tab = reinterpret_cast<float *>(lds);
    const float *src = table + (int64_t)chunk * depth * kBinFeatures;
    for (int i = tid; i < depth * kBinFeatures; i += kBinWaves * 64) tab[i] = src[i];
  }
  __syncthreads(); // the only block-wide barrier: from here on the waves run on their own
  unsigned char *stage = lds + tableBytes + (uint32_t)wave * (64u * kBinLaneStride);
  unsigned char *mine = stage + lane * kBinLaneStride;
  const int64_t numRowBlocks = (rows + kBinRows - 1) / kBinRows;
  const int64_t rbBegin = rowGroup * rowBlocksPerBlock; // (past the end for the padding blocks of the last 8 groups)
  const int64_t rbEnd = rbBegin + rowBlocksPerBlock < numRowBlocks ? rbBegin + rowBlocksPerBlock : numRowBlocks;
  const int fClamped = f < F ? f : F - 1;
  const uint32_t laneBytes = (uint32_t)lane * 4u;
  // The rows of the next pass are requested before the current pass is searched (two register
  // buffers), so that the wave always has loads in flight.
  float va[kBinRowsPerPass], vb[kBinRowsPerPass];
  int64_t rb = rbBegin + wave;
  if (rb < rbEnd) BinLoadRows(x, rows, F, fClamped, rb * kBinRows, va);
  for (; rb < rbEnd; rb += kBinWaves) {
    const int64_t rowBase = rb * kBinRows;
    BinLoadRows(x, rows, F, fClamped, rowBase + kBinRowsPerPass, vb);
    BinSearchRows<kLevels>(va, laneBytes, mine);
    BinLoadRows(x, rows, F, fClamped, rowBase + 2 * kBinRowsPerPass, va);
    BinSearchRows<kLevels>(vb, laneBytes, mine + 16);
    BinLoadRows(x, rows, F, fClamped, rowBase + 3 * kBinRowsPerPass, vb);
    BinSearchRows<kLevels>(va, laneBytes, mine + 32);
    const int64_t rbNext = rb + kBinWaves < rbEnd ? rb + kBinWaves : rb; // (the last block re-reads its own rows)
    BinLoadRows(x, rows, F, fClamped, rbNext * kBinRows, va);
    BinSearchRows<kLevels>(vb, laneBytes, mine + 48);
    // the wave's 64 features x 64 rows leave as contiguous 16-byte pieces (piece = feature * 4 + pass)
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    uint8_t *dst = ranks + (rb * F + f0) * kBinRows;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int piece = j * 64 + lane;
      const Piece value = *reinterpret_cast<const Piece *>(stage + (piece >> 2) * kBinLaneStride + (piece & 3) * 16);
      if (f0 + (piece >> 2) < F) *reinterpret_cast<Piece *>(dst + piece * 16) = value;
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier(); // the staging area is rewritten by the next row block
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }
}

// ---------------------------------------------------------------------------
// Two-byte ranks for narrow models.  For every (row, feature) the kernel counts how many of the feature's
// sorted distinct split thresholds are <= the value and writes the count as 16 bits into the tile layout the
// row-parallel kernel copies verbatim: [block of RB rows][feature pair][row][2] (the two ranks of a pair share
// a dword, so a row's LDS column keeps one bank of its own).  NaN and +inf count every entry of the table (a
// rank above every node's threshold index: they go right at every node, as the f32 compare sends them).  The
// slots of the pad feature (and of the unused half of an odd last pair) get rank 0.
//
// A block owns one chunk of feature pairs, whose threshold tables sit in LDS, and a range of rows, which it
// takes 1024 at a time: the chunk's columns of those rows are read with row-contiguous loads and left
// transposed in LDS (a lane that walked its row's columns in global memory would touch a cache line per load
// and evict it before the next: measured 1.2 to 2 times slower), then a lane is a row: it picks its values out
// of its own LDS bank and searches one feature after the other.  Every table is a complete search tree in
// breadth-first order (entry 0 the root, then its children, ...) and the feature is the same for the whole
// wave, so at search step l the lanes read among 2^l neighbouring entries (one bank each up to 64, broadcast
// where they meet).  Blocks 8 apart in launch order (same XCD, back to back) take the chunks of one row range,
// so that the cache lines of a row, which the chunks share, are fetched from HBM once.
// ---------------------------------------------------------------------------
// (measured on configurations 2, 3 and 5 at 2^20 rows: 16 waves x 1 group 0.105 / 0.169 / 0.290 ms, 8 x 2 0.120 / 0.189 /
// 0.310, 4 x 4 0.152 / 0.252 / 0.365: the two phases of a tile are latency-bound, and waves hide latency better
// than chains do)
constexpr int kRankWaves = 16;
constexpr int kRankChains = 1;                              // 64-row groups a lane searches side by side
constexpr int kRankTileRows = kRankWaves * kRankChains * 64; // rows a block ranks between two barriers
constexpr int kRankStride = kRankTileRows + 1;              // floats per feature column of the staging tile
constexpr int kRankLoads = 8;                               // loads a lane keeps in flight while staging

__global__ void __launch_bounds__(kRankWaves * 64)
RankRows16Kernel(const float *__restrict__ x, const float *__restrict__ tables, const RankFeatureDesc *__restrict__ features,
                 const RankChunkDesc *__restrict__ chunks, uint32_t *__restrict__ ranks, int64_t rows, int F, int RB,
                 int numChunks, int tilesPerBlock, int64_t rowTiles, uint32_t tableRegionBytes) {
  extern __shared__ __align__(16) unsigned char lds[];
  const uint32_t linear = blockIdx.x;
  const int chunk = (int)((linear >> 3) % (uint32_t)numChunks);
  const int64_t range = (int64_t)(linear & 7u) + 8 * (int64_t)(linear / (8u * (uint32_t)numChunks));
  const RankChunkDesc ck = chunks[chunk];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  constexpr int threads = kRankWaves * 64;
  {
    float *tab = reinterpret_cast<float *>(lds);
    const float *src = tables + ck.tableBegin;
    for (uint32_t i = tid; i < ck.tableEntries; i += threads) tab[i] = src[i];
  }
  float *stage = reinterpret_cast<float *>(lds + tableRegionBytes); // [feature of the chunk][kRankStride]
  const uint32_t stageAddress = tableRegionBytes;
  const int pairsTotal = (F + 2) >> 1;
  const int Fc = (int)ck.numFeatures;                                // slots of the chunk (whole pairs)
  const int live = (int)ck.firstFeature + Fc <= F ? Fc : F - (int)ck.firstFeature; // of which real features (may be <= 0)
  const float invLive = live > 0 ? 1.0f / (float)live : 0.0f;
  const int64_t tBegin = range * tilesPerBlock; // (past the end for the padding blocks of the last 8 ranges)
  const int64_t tEnd = tBegin + tilesPerBlock < rowTiles ? tBegin + tilesPerBlock : rowTiles;
  for (int64_t tile = tBegin; tile < tEnd; ++tile) {
    const int64_t row0 = tile * kRankTileRows;
    __syncthreads(); // tables loaded / the staging tile is no longer read
    // The chunk's columns of the tile's rows: element e = (row, column) in row-major order, so that a wave's load
    // covers whole row segments; rows past the batch (padding of the last row block) take the last row's values.
    const int total = kRankTileRows * live;
    for (int e0 = tid; e0 < total; e0 += threads * kRankLoads) {
      float value[kRankLoads];
      int where[kRankLoads];
#pragma unroll
      for (int u = 0; u < kRankLoads; ++u) {
        const int e = e0 + u * threads < total ? e0 + u * threads : total - 1;
        int r = (int)((float)e * invLive);
        if (r * live > e) --r;
        if ((r + 1) * live <= e) ++r;
        const int j = e - r * live;
        const int64_t row = row0 + r < rows ? row0 + r : rows - 1;
        value[u] = x[row * F + ck.firstFeature + j];
        where[u] = j * kRankStride + r;
      }
#pragma unroll
      for (int u = 0; u < kRankLoads; ++u)
        if (e0 + u * threads < total) stage[where[u]] = value[u];
    }
    __syncthreads();
    // a lane is a row in each of its wave's kRankChains groups of 64 rows
    const int r0 = wave * (kRankChains * 64) + lane;
    int64_t slot[kRankChains];
#pragma unroll
    for (int c = 0; c < kRankChains; ++c) {
      const int64_t row = row0 + r0 + c * 64;
      slot[c] = (row / RB) * (int64_t)pairsTotal * RB + (row % RB) + (int64_t)(ck.firstFeature >> 1) * RB;
    }
    for (int j0 = 0; j0 < Fc; j0 += 2) {
      uint32_t rank[2][kRankChains];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int j = j0 + h;
        if (j >= live) { // the pad feature's slot and the unused half of an odd last pair
#pragma unroll
          for (int c = 0; c < kRankChains; ++c) rank[h][c] = 0;
          continue;
        }
        const RankFeatureDesc fd = features[ck.firstFeature + j]; // (the same for the whole wave)
        const uint32_t base = fd.tableOffset * 4u;                 // LDS byte address of the table's root
        const uint32_t goLeft = 4u - base, goRight = 8u - base;
        float v[kRankChains];
        uint32_t pos[kRankChains];
#pragma unroll
        for (int c = 0; c < kRankChains; ++c) {
          v[c] = LdsLoadFloat(stageAddress + (uint32_t)(j * kRankStride + r0 + c * 64) * 4u);
          pos[c] = base;
        }
        for (uint32_t level = 0; level < fd.levels; ++level) {
          float probe[kRankChains];
#pragma unroll
          for (int c = 0; c < kRankChains; ++c) probe[c] = LdsLoadFloat(pos[c]);
#pragma unroll
          for (int c = 0; c < kRankChains; ++c) pos[c] = (pos[c] << 1) + (v[c] < probe[c] ? goLeft : goRight); // NaN: right at every step
        }
        // entry index reached below the last table level, minus the 2^levels - 1 entries of the table = thresholds <= value
        const uint32_t entries = (1u << fd.levels) - 1u;
#pragma unroll
        for (int c = 0; c < kRankChains; ++c) rank[h][c] = ((pos[c] - base) >> 2) - entries;
      }
#pragma unroll
      for (int c = 0; c < kRankChains; ++c) ranks[slot[c] + (int64_t)(j0 >> 1) * RB] = rank[0][c] | (rank[1][c] << 16);
    }
  }
}

// ---------------------------------------------------------------------------
// Sums the tree-slice partials of each row (in slice order, starting from the
// initial value), then applies the output transform.  Multiclass rows get the
// arg-max of the f32 per-class sums with the generated-code tie rule (running
// maximum replaced unless strictly greater, so ties go to the larger class id;
// src/mlir/LowerReduceOps.cpp:148-187) and, on request, the sums and their
// softmax.
// ---------------------------------------------------------------------------
// A row's class sums -> class id (arg-max of the f32 sums, ties to the larger id) and, on request, the f32 sums and
// their softmax.
template <typename SumOf> // class -> its sum
__device__ __forceinline__ void FinishClasses(SumOf sumOf, int C, int64_t row, float *out, int8_t *classOut, float *margins,
                                              float *probabilities) {
  float best = -INFINITY;
  int bestClass = 0;
  double maxMargin = -INFINITY;
  for (int c = 0; c < C; ++c) {
    const double sum = sumOf(c);
    const float m = (float)sum;
    if (margins) margins[row * C + c] = m;
    if (!(best > m)) { best = m; bestClass = c; }
    maxMargin = sum > maxMargin ? sum : maxMargin;
  }
  if (classOut) classOut[row] = (int8_t)bestClass;
  if (out) out[row] = (float)bestClass;
  if (probabilities) {
    double z = 0.0;
    for (int c = 0; c < C; ++c) z += exp(sumOf(c) - maxMargin);
    for (int c = 0; c < C; ++c) probabilities[row * C + c] = (float)(exp(sumOf(c) - maxMargin) / z);
  }
}

// How many slots of the partial sums hold parts of a row.
__device__ __forceinline__ int PartsOfRow(const FinalizeParams &p, int64_t row) {
  if (p.splitBlocks == 0) return p.treeSlices;
  return SplitLine{((p.rows + p.rowsPerBlock - 1) / p.rowsPerBlock) * p.groups, p.groups, p.splitBlocks}.Parts(row / p.rowsPerBlock);
}

__global__ void __launch_bounds__(256) FinalizeKernel(const FinalizeParams p) {
  const int64_t row = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (row >= p.rows) return;
  const int parts = PartsOfRow(p, row);
  double margin = p.initialValue;
#pragma unroll 4
  for (int s = 0; s < parts; ++s) margin += p.partial[(int64_t)s * p.rows + row];
  p.out[row] = (float)(p.transform == 1 ? 1.0 / (1.0 + exp(-margin)) : margin);
}

// Classifiers: the block's rows x classes are read as they lie (coalesced; a lane per row read a line per class and all
// of them three times: 13 us for 65537 rows x 8 classes x 2 slices), meet in LDS, and the rows are finished there.  A sum per
// lane (more in large batches): blocks of 128 rows, whose lanes wait for memory four times in a row, took 65537 rows x 8 classes
// 4.7 us longer with sums and softmax.  With twelve parts and more to add, two groups of 256 lanes take every second of them:
// class ids of 900 trees, 1400 rows x 5 classes in 40 parts 18.2 us with one group and 16.9 with two, 1800 x 8 in 23 15.0 and
// 14.6, 4380 x 8 in twelve 16.0 and 15.6; but 6000 x 3 in ten 15.0 and 15.6, 25000 x 9 in ten 41.5 and 43.9, 45000 x 6 in four 48.1
// and 50.1, 80000 x 13 in up to five 94.6 and 99.9.
constexpr int kFinalizeLds = 4096; // doubles of sums a block holds
constexpr int kClassPartsShared = 12;

__global__ void __launch_bounds__(1024) FinalizeClassesKernel(const FinalizeParams p, int rowsPerBlock) {
  extern __shared__ __align__(16) unsigned char lds[];
  double *sums = reinterpret_cast<double *>(lds); // [row][class], rows an odd number of doubles apart
  const int C = p.numClasses, stride = C | 1;
  double *rowMax = sums + rowsPerBlock * stride, *rowZ = rowMax + rowsPerBlock, *others = rowZ + rowsPerBlock;
  const int64_t row0 = (int64_t)blockIdx.x * rowsPerBlock;
  const int valid = p.rows - row0 < rowsPerBlock ? (int)(p.rows - row0) : rowsPerBlock;
  const int tid = threadIdx.x, threads = blockDim.x;
  const int groups = threads >> 8, group = __builtin_amdgcn_readfirstlane(tid >> 8);
  const int64_t slot = p.rows * C;
  double *mine = group == 0 ? sums : others + (group - 1) * (rowsPerBlock * stride);
  for (int e = tid & 255; e < valid * C; e += 256) {
    const int r = e / C, c = e - r * C;
    // (a group's first two parts are on their way while the divisions that count the parts run; a slot is there, filled or not)
    const double *at = p.partial + row0 * C + e;
    const double first = at[group * slot], second = group + groups < p.treeSlices ? at[(group + groups) * slot] : 0.0;
    const int parts = PartsOfRow(p, row0 + r);
    double sum = group == 0 ? p.initialValue : 0.0;
    if (group < parts) sum += first;
    if (group + groups < parts) sum += second;
#pragma unroll 4
    for (int s = group + 2 * groups; s < parts; s += groups) sum += at[s * slot];
    mine[r * stride + c] = sum;
    if (groups == 1 && p.margins) p.margins[row0 * C + e] = (float)sum;
  }
  if (groups > 1) {
    __syncthreads();
    for (int e = tid; e < valid * C; e += threads) {
      const int r = e / C, c = e - r * C;
      double sum = sums[r * stride + c];
      for (int g = 1; g < groups; ++g) sum += others[(g - 1) * (rowsPerBlock * stride) + r * stride + c];
      sums[r * stride + c] = sum;
      if (p.margins) p.margins[row0 * C + e] = (float)sum;
    }
  }
  __syncthreads();
  for (int r = tid; r < valid; r += threads) {
    float best = -INFINITY;
    int bestClass = 0;
    double maxMargin = -INFINITY;
    for (int c = 0; c < C; ++c) {
      const double margin = sums[r * stride + c];
      const float m = (float)margin;
      if (!(best > m)) { best = m; bestClass = c; }
      maxMargin = margin > maxMargin ? margin : maxMargin;
    }
    if (p.classOut) p.classOut[row0 + r] = (int8_t)bestClass;
    if (p.out) p.out[row0 + r] = (float)bestClass;
    rowMax[r] = maxMargin;
  }
  if (!p.probabilities) return;
  __syncthreads();
  for (int e = tid; e < valid * C; e += threads) {
    const int r = e / C, at = r * stride + (e - r * C);
    sums[at] = exp(sums[at] - rowMax[r]);
  }
  __syncthreads();
  for (int r = tid; r < valid; r += threads) {
    double z = 0.0;
    for (int c = 0; c < C; ++c) z += sums[r * stride + c];
    rowZ[r] = z;
  }
  __syncthreads();
  for (int e = tid; e < valid * C; e += threads) {
    const int r = e / C;
    p.probabilities[row0 * C + e] = (float)(sums[r * stride + (e - r * C)] / rowZ[r]);
  }
}

// More classes than a block's LDS holds sums of: a lane per row adds the parts again each time a sum is needed.
__global__ void __launch_bounds__(256) FinalizeManyClassesKernel(const FinalizeParams p) {
  const int64_t row = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (row >= p.rows) return;
  const int parts = PartsOfRow(p, row);
  FinishClasses(
      [&](int c) {
        double margin = p.initialValue;
        for (int s = 0; s < parts; ++s) margin += p.partial[((int64_t)s * p.rows + row) * p.numClasses + c];
        return margin;
      },
      p.numClasses, row, p.out, p.classOut, p.margins, p.probabilities);
}

// Small batches split over several tree slices: 64 rows a block, a lane each, and its waves share the slices, so that a lane
// waits for few loads and a wave reads 512 contiguous bytes.  (A wave per sum, lanes along the slices, read a 64-byte piece of
// memory for each of its 8 bytes: 4096 rows x 32 slices 3.0 us, 2.5 here; the call 15.1 and 13.9.)  Each wave adds its slices
// in slice order, the waves are added in order: the order of additions depends on the number of slices alone.  Calls that way and
// with a lane per row, 2000 to 66000 rows: two to five slices the same within 4 % either way (13744 rows in four 10.4 and 10.2 us,
// 26518 17.5 and 16.8), six 2 % less (10042 rows 10.2 and 10.4), ten 6 to 8 % (6233 12.5 and 13.6), twenty 6 to 13 %.
constexpr int kWideFinalizeSlices = 6;
constexpr int64_t kWideFinalizeRows = 65536;

template <int kWaves> // 4, or 8 from so many slices on
__global__ void __launch_bounds__(kWaves * 64) FinalizeWideKernel(const FinalizeParams p) {
  __shared__ double meet[kWaves][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t row = (int64_t)blockIdx.x * 64 + lane;
  if (row < p.rows) {
    const int parts = PartsOfRow(p, row);
    double sum = 0.0;
#pragma unroll 4
    for (int s = wave; s < parts; s += kWaves) sum += p.partial[(int64_t)s * p.rows + row];
    meet[wave][lane] = sum;
  }
  __syncthreads();
  if (wave != 0 || row >= p.rows) return;
  double sum = meet[0][lane];
  for (int w = 1; w < kWaves; ++w) sum += meet[w][lane];
  const double margin = p.initialValue + sum;
  p.out[row] = (float)(p.transform == 1 ? 1.0 / (1.0 + exp(-margin)) : margin);
}

// ---------------------------------------------------------------------------
// A few rows: one launch, one lane per (row, tree).  What such a batch waits for is latency - of the launches, of
// staging tree groups in LDS and of the dependent node reads - so nothing is staged but the rows and nothing is left
// to a second kernel: a lane reads a tree three levels at a time (one 48-byte block, three 16-byte loads in flight
// together, so a walk of 8 levels waits for three loads of L2 latency instead of nine), leaves its leaf value in LDS,
// and a wave per (row, class) adds them in a fixed order.  One row through 1000 trees of depth 8 took 15.2 us a call
// with the tree-parallel kernel and its finalize launch, 6.5 here (4.4 of them the kernel).
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(1024) FewRowsKernel(const FewRowsParams p, int rowsPerBlock, int leafStride) {
  extern __shared__ __align__(16) unsigned char lds[];
  const int tid = threadIdx.x, threads = blockDim.x;
  const int T = p.numTrees, F = p.numFeatures, R = rowsPerBlock;
  const int Cn = p.numClasses > 0 ? p.numClasses : 1;
  const int64_t row0 = (int64_t)blockIdx.x * R;
  const int valid = p.rows - row0 < R ? (int)(p.rows - row0) : R;
  float *leaves = reinterpret_cast<float *>(lds);
  float *rowTile = leaves + (size_t)T * leafStride;
  double *sums = reinterpret_cast<double *>((reinterpret_cast<uintptr_t>(rowTile + (size_t)R * F) + 7) & ~(uintptr_t)7);
  const U32x4 *blocks = reinterpret_cast<const U32x4 *>(p.blocks);
  const int items = valid * T; // item i: row i % valid of tree i / valid (lanes of a wave share the top of a tree)

  // the first trees' top blocks are requested before the rows are staged
  U32x4 q0{}, q1{}, q2{};
  if (tid < items) {
    const U32x4 *b = blocks + (size_t)(tid / valid) * 3;
    q0 = b[0], q1 = b[1], q2 = b[2];
  }
  {
    const float *src = p.x + row0 * F;
    for (int e = tid; e < valid * F; e += threads) rowTile[e] = src[e];
  }
  __syncthreads();
  for (int i = tid; i < items; i += threads) {
    const int t = i / valid, r = i - t * valid;
    const float *row = rowTile + r * F;
    if (i != tid) {
      const U32x4 *b = blocks + (size_t)t * 3;
      q0 = b[0], q1 = b[1], q2 = b[2];
    }
    float leaf;
    for (;;) {
      const uint32_t f0 = q2.x & 0xFFFFu;
      leaf = AsFloat(q0.x);
      if (f0 == kFewRowsLeaf) break;
      const bool right0 = !(row[f0] < leaf); // (NaN goes right)
      const uint32_t f1 = right0 ? q2.y & 0xFFFFu : q2.x >> 16;
      leaf = AsFloat(right0 ? q0.z : q0.y);
      if (f1 == kFewRowsLeaf) break;
      const bool right1 = !(row[f1] < leaf);
      const uint32_t pair = right0 ? (q2.w << 16) | (q2.z >> 16) : (q2.z << 16) | (q2.y >> 16); // features of slots 3, 4 or 5, 6
      const uint32_t f2 = right1 ? pair >> 16 : pair & 0xFFFFu;
      leaf = AsFloat(right0 ? (right1 ? q1.z : q1.y) : (right1 ? q1.x : q0.w));
      if (f2 == kFewRowsLeaf) break;
      const bool right2 = !(row[f2] < leaf);
      const uint32_t exit = (right0 ? 4u : 0u) + (right1 ? 2u : 0u) + (right2 ? 1u : 0u);
      const uint32_t child = q1.w + (uint32_t)__popc((q2.w >> 16) & ((1u << exit) - 1u));
      const U32x4 *b = blocks + (size_t)child * 3;
      q0 = b[0], q1 = b[1], q2 = b[2];
    }
    leaves[(size_t)t * leafStride + r] = leaf;
  }
  __syncthreads();
  // a wave per (row, class): lanes take trees in turn, a butterfly adds the lanes
  const int lane = tid & 63;
  for (int pair = tid >> 6; pair < valid * Cn; pair += threads >> 6) {
    const int r = pair / Cn, c = pair - r * Cn;
    const int end = p.numClasses > 0 ? p.classBegin[c + 1] : T;
    double sum = 0.0;
    for (int t = (p.numClasses > 0 ? p.classBegin[c] : 0) + lane; t < end; t += 64) sum += (double)leaves[(size_t)t * leafStride + r];
    for (int m = 1; m <= 32; m <<= 1) sum += ShuffleXor(sum, m); // (ascending: see ShuffleXor)
    const double margin = p.initialValue + sum;
    if (lane != 0) continue;
    if (p.numClasses == 0) p.out[row0 + r] = (float)(p.transform == 1 ? 1.0 / (1.0 + exp(-margin)) : margin);
    else sums[pair] = margin;
  }
  if (p.numClasses == 0) return;
  __syncthreads();
  for (int r = tid; r < valid; r += threads)
    FinishClasses([&](int c) { return sums[r * Cn + c]; }, Cn, row0 + r, p.out, p.classOut, p.margins, p.probabilities);
}

// Address of the two children of a stream's word: the pair's index is the word's third byte, eight bytes a pair, from `tree` on.
// (A sum of four byte products and the third operand: one instruction for the two
// that pick the byte and add it: 262144 rows x 2000 features, 1000 trees 1226 -> 1190 us.)
__device__ __forceinline__ uint32_t StreamChildren(uint32_t word, uint32_t tree) {
  return __builtin_amdgcn_udot4(word, 0x00080000u, tree, false);
}

// ---------------------------------------------------------------------------
// Wide rows, rank-quantised: a block keeps 32 rows of one byte per feature in LDS (64 KB at 2000 features) and every
// wave streams its own bundles of eight trees through 8 KB of its own, two bundles deep: while one is walked the next is
// on its way from L2 (direct global -> LDS loads), so no wave waits for a copy or for another wave - the tree groups of
// the row-parallel kernel, which all waves of a block copy, wait for and walk together with nothing else on the CU to
// cover it, kept the LDS pipes 37 % busy.  The two halves of a wave walk different trees over the same 32 rows, each lane
// four chains (two, in bundles of four trees, where bigger trees leave bundles of eight short); 32 rows instead of 64
// leave the room (twelve waves x two buffers), and 4-byte nodes halve what a bundle takes: a step is a 4-byte node read
// and a one-byte rank read.  Leaf values stay in global memory, one gather per tree, issued a bundle ahead of its use.
//
// With three waves a SIMD every wait in a wave's chain is seen.  So: the lane holds the word it stands on and reads both
// children (8 bytes side by side, at the price of 4) together with the rank, one LDS round trip a level instead of two; a
// bundle's depth and its trees' roots stand in the head of its image, its place comes through a vector load (a scalar load took
// its latency every bundle); chains ask for their next level two by two, while the other two's reads are on their way; and a
// workgroup stays, with the next rows' ranks on their way to registers while its last bundle is walked (it
// has its compute unit's LDS to itself: nothing else walks while it loads).  Whole calls of 262144 rows x 2000 features, 1000
// trees of depth 8: 1308 us with two trips a level and a workgroup per 32 rows, 1223 with one trip and workgroups that stay, 1190
// with one instruction to a child's address (StreamChildren), 1152 with the roots in the heads and chains that wait for their
// own reads only, 1131 with chains two by two (fewer instructions between the waits and the next reads; all four at once 1190), 1114 with
// their compares and addresses ordered so that no instruction waits for the one before.
// ---------------------------------------------------------------------------
// kStays: workgroups go on with other rows.  Where none does, what that takes (76 VGPRs and 1700 bytes of code) is left out: 3644
// rows x 167 trees of 896 features 16.8 -> 16.2 us, 5504 x 92 of 1401 21.7 -> 21.2, 7713 x 46 of 672 15.2 -> 14.5.
template <int K, bool kStays> // chains
__global__ void __launch_bounds__(kStreamMaxWaves * 64)
RankStreamKernel(const uint8_t *__restrict__ ranks, const uint32_t *__restrict__ words, const float *__restrict__ values,
                 const uint32_t *__restrict__ bundles, int64_t rows, int F, int numBundles, int slices, int transform,
                 double initialValue, float *__restrict__ out, double *__restrict__ partial) {
  extern __shared__ __align__(16) unsigned char lds[]; // [feature][32 rows] ranks, pad feature included | two bundles per wave
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int waves = blockDim.x >> 6;
  // The two halves of a 64-row rank tile share its cache lines: their blocks are 8 apart in launch order (same XCD).
  const auto blockOf = [](uint32_t linear) { return (int64_t)(linear >> 4) * 16 + (int64_t)((linear & 7u) * 2u + ((linear >> 3) & 1u)); };
  const uint32_t padded = (uint32_t)((rows + 16 * kStreamRows - 1) / (16 * kStreamRows)) * 16u;
  const auto blockFrom = [&](uint32_t linear) { // the first that has rows, of those this workgroup takes
    while (linear < padded && blockOf(linear) * kStreamRows >= rows) linear = kStays ? linear + gridDim.x : padded;
    return linear;
  };
  uint32_t linear = blockFrom(blockIdx.x);
  if (linear >= padded) return;
  const uint32_t tileBytes = ((uint32_t)(F + 1) * kStreamRows + 15u) & ~15u;
  const uint32_t mine = tileBytes + (uint32_t)wave * (2u * kStreamBundleBytes); // this wave's two bundles
  const int pieces = F * 2; // of a row block's ranks: piece p is half (p & 1) of the 32 bytes of feature p / 2
  // (A uniform base and 32 bits of offset: with 64-bit addresses per lane the kernel spilled two registers to scratch memory.  5504
  // rows x 92 trees 20.4 -> 20.1 us, 20129 x 656 56.4 -> 54.8, 100000 x 300 207.5 -> 204.1; 262144 x 1000 1211 -> 1225.)
  const auto pieceOf = [&](uint32_t of, int p) {
    const int64_t block = blockOf(of);
    const uint8_t *base = ranks + (block >> 1) * F * 64 + (block & 1) * kStreamRows;
    return base + ((uint32_t)(p >> 1) * 64u + (uint32_t)(p & 1) * 16u);
  };
  // 16 bytes per lane to LDS address DST + 16 * lane.  (Not the builtin: while one of those is outstanding the compiler
  // awaits LDS reads only all together, and here one nearly always is.  The waits for these copies are the explicit ones.)
#define TBAMD_STREAM_COPY(SRC, DST)                                                                                    \
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(SRC), "s"(DST) : "memory", "m0");
  for (int p0 = wave * 64; p0 < pieces; p0 += waves * 64)
    if (p0 + lane < pieces) TBAMD_STREAM_COPY(pieceOf(linear, p0 + lane), (uint32_t)p0 * 16u)
  if (tid < kStreamRows / 4) *reinterpret_cast<uint32_t *>(lds + (uint32_t)F * kStreamRows + tid * 4) = 0; // pad feature
  const int first = (int)((int64_t)numBundles * blockIdx.y / slices), last = (int)((int64_t)numBundles * (blockIdx.y + 1) / slices);
#define TBAMD_STREAM_BUNDLE(BEGIN, BUFFER)                                                                             \
  {                                                                                                                    \
    const U32x4 *src = reinterpret_cast<const U32x4 *>(words + (BEGIN)) + lane;                                        \
    _Pragma("unroll") for (uint32_t q = 0; q < kStreamBundleBytes; q += 1024u)                                         \
        TBAMD_STREAM_COPY(src + q / 16u, (BUFFER) + q)                                                                 \
  }
  // The bundle walked next, and the one behind it; behind the last one comes the first, for the next row block.
  const int begin = first + wave;
  const auto after = [&](int b) { return b + waves < last ? b + waves : begin; };
  // (The places of the bundles come through vector loads, a bundle ahead: a scalar load in flight would make every LDS read's
  // wait one for it.  What else is to be known of a bundle stands in its image.)
  uint32_t zero;
  asm volatile("v_mov_b32 %0, 0" : "=v"(zero));
  uint32_t nextBegin = 0;
  if (begin < last) {
    const uint32_t now = bundles[begin];
    TBAMD_STREAM_BUNDLE(now, mine)
    nextBegin = bundles[(uint32_t)after(begin) + zero];
  }
  // Bundles of wave w, per row block.  (One division, while the copies are on their way: one for every wave's sum, when a row
  // block ends, took 0.4 to 0.8 us of each: 217490 rows x 107 trees of 673 features 274 -> 254 us.)
  const int everyWave = kStays ? (last - first) / waves : 0, waveMore = (last - first) - everyWave * waves;
  const auto bundlesOf = [&](int w) { return everyWave + (w < waveMore ? 1 : 0); };
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads(); // the rows are there; until they are through, the waves run on their own

  const uint32_t row = (uint32_t)lane & 31u;
  const bool upper = lane >= 32;
  uint32_t buffer = mine;
  for (uint32_t pass = 0;; ++pass) {
    const uint32_t nextLinear = kStays ? blockFrom(linear + gridDim.x) : padded;
    const bool more = kStays && nextLinear < padded;
    U32x4 nextRanks[kStreamTilePieces];
#define TBAMD_STREAM_NEXT_ROWS                                                                                         \
  _Pragma("unroll") for (int i = 0; i < kStreamTilePieces; ++i) {                                                      \
    const int p = (i * waves + wave) * 64 + lane;                                                                      \
    nextRanks[i] = *reinterpret_cast<const U32x4 *>(pieceOf(nextLinear, p < pieces ? p : pieces - 1));                 \
  }
    double acc = 0.0;
    float leaf[K];
    uint32_t at[K]; // where the leaf values of the bundle before lie (entry 0: none)
#pragma unroll
    for (int k = 0; k < K; ++k) leaf[k] = 0.0f, at[k] = 0u;
    if (begin >= last && more) TBAMD_STREAM_NEXT_ROWS
    for (int b = begin; b < last; b += waves) {
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); // this bundle, and the leaf values of the one before the last
      const uint32_t follows = __builtin_amdgcn_readfirstlane(nextBegin);
#pragma unroll
      for (int k = 0; k < K; ++k) acc += (double)leaf[k];
#pragma unroll
      for (int k = 0; k < K; ++k) leaf[k] = values[at[k]];
      const uint32_t other = buffer == mine ? mine + kStreamBundleBytes : mine;
      if (b + waves < last || more) TBAMD_STREAM_BUNDLE(follows, other)
      nextBegin = bundles[(uint32_t)after(after(b)) + zero];
      if (b + waves >= last && more) TBAMD_STREAM_NEXT_ROWS
      const uint32_t headAt = buffer + (upper ? (uint32_t)sizeof(DeviceStreamHead) : 0u);
      const U32x4 head = LdsLoadQuad(headAt), rootWords = LdsLoadQuad(headAt + 16u), valueBegin = LdsLoadQuad(headAt + 32u);
      const int depth = (int)__builtin_amdgcn_readfirstlane(head.z);
      uint32_t tree[K], node[K]; // where the words of a tree lie, and the word the lane stands on
#pragma unroll
      for (int k = 0; k < K; ++k) {
        tree[k] = buffer + (k & 1 ? head[k / 2] >> 16 : head[k / 2] & 0xFFFFu);
        node[k] = rootWords[k];
      }
      // Two chains ask for their next level as soon as their own reads are there, the others' still on their way.  (Left to itself
      // the compiler waits for all chains before the first compares, and reads one child, when the rank is there.)
      U32x2 children[K];
      uint32_t rank[K];
      const auto ask = [&](int k, bool both) {
        uint32_t below[2], at[2];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          below[i] = both ? StreamChildren(node[k + i], tree[k + i]) : 0u;
          at[i] = AddChild(node[k + i], row);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < 2; ++i) rank[k + i] = LdsLoadByte(at[i]);
        if (both) {
#pragma unroll
          for (int i = 0; i < 2; ++i) children[k + i] = LdsLoadNode(below[i]);
        }
      };
      const auto step = [&](int k) {
        uint64_t second; // (a mask may be read two instructions after it is written: the second compare stands in the first one's wait)
        asm("v_cmp_lt_u32_sdwa vcc, %3, %0 src0_sel:DWORD src1_sel:BYTE_3\n\t"
            "v_cmp_lt_u32_sdwa %2, %4, %1 src0_sel:DWORD src1_sel:BYTE_3\n\t"
            "s_nop 0\n\t"
            "v_cndmask_b32_e32 %0, %6, %5, vcc\n\t"
            "v_cndmask_b32_e64 %1, %8, %7, %2"
            : "+&v"(node[k]), "+&v"(node[k + 1]), "=&s"(second)
            : "v"(rank[k]), "v"(rank[k + 1]), "v"(children[k].x), "v"(children[k].y), "v"(children[k + 1].x), "v"(children[k + 1].y)
            : "vcc");
      };
      if (depth > 1) {
#pragma unroll
        for (int k = 0; k < K; k += 2) ask(k, true);
        for (int d = 2; d < depth; ++d) {
#pragma unroll
          for (int k = 0; k < K; k += 2) {
            __builtin_amdgcn_sched_barrier(0);
            step(k);
            ask(k, true);
          }
        }
#pragma unroll
        for (int k = 0; k < K; k += 2) {
          __builtin_amdgcn_sched_barrier(0);
          step(k);
          ask(k, false); // (the last level's words are not there: only which they are counts)
        }
      } else {
#pragma unroll
        for (int k = 0; k < K; k += 2) ask(k, false);
      }
#pragma unroll
      for (int k = 0; k < K; ++k) at[k] = valueBegin[k] + ((node[k] >> 15) & 0x1FEu) + (rank[k] < (node[k] >> 24) ? 0u : 1u);
      buffer = other;
    }
#pragma unroll
    for (int k = 0; k < K; ++k) acc += (double)leaf[k];
#pragma unroll
    for (int k = 0; k < K; ++k) acc += (double)values[at[k]];
    acc += ShuffleXor(acc, 32);
    // A wave's sums go where its last bundle was: its other buffer may hold the first one for the next rows.  (Of a workgroup
    // that does not stay no copy is on its way any more: either buffer.)
    const auto meetOf = [&](int w) {
      const uint32_t walked = kStays ? (uint32_t)bundlesOf(w) * (pass + 1u) : 0u;
      return reinterpret_cast<double *>(lds + tileBytes + (uint32_t)w * (2u * kStreamBundleBytes) + (walked & 1u ? 0u : kStreamBundleBytes));
    };
    if (lane < kStreamRows) meetOf(wave)[lane] = acc;
    __syncthreads(); // the sums are there, nobody reads ranks any more
    if (more) {
#pragma unroll
      for (int i = 0; i < kStreamTilePieces; ++i) {
        const int p = (i * waves + wave) * 64 + lane;
        if (p < pieces) *reinterpret_cast<U32x4 *>(lds + (uint32_t)p * 16u) = nextRanks[i];
      }
    }
    const int64_t r = blockOf(linear) * kStreamRows + tid;
    if (tid < kStreamRows && r < rows) {
      double sum = 0.0;
      for (int w = 0; w < waves; ++w) sum += meetOf(w)[tid];
      if (partial) {
        partial[(int64_t)blockIdx.y * rows + r] = sum;
      } else {
        const double margin = initialValue + sum;
        out[r] = (float)(transform == 1 ? 1.0 / (1.0 + exp(-margin)) : margin);
      }
    }
    if (!more) return;
    __syncthreads(); // the next rows are there, the sums are read
    linear = nextLinear;
  }
#undef TBAMD_STREAM_NEXT_ROWS
#undef TBAMD_STREAM_BUNDLE
#undef TBAMD_STREAM_COPY
}

// The ceiling on dynamic LDS is an attribute of each kernel on each device: it is raised once per kernel and
// device, to the whole 160 KB, instead of on every launch (a runtime call that small batches would pay for each
// time).  Two threads that meet here for the first time both make the call, which is harmless.
template <auto Kernel> hipError_t AllowFullLds() {
  constexpr int kMaxDevices = 64;
  static std::atomic<bool> raised[kMaxDevices];
  int device = 0;
  hipError_t e = hipGetDevice(&device);
  if (e != hipSuccess) return e;
  if (device >= 0 && device < kMaxDevices && raised[device].load(std::memory_order_acquire)) return hipSuccess;
  e = hipFuncSetAttribute(reinterpret_cast<const void *>(Kernel), hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
  if (e == hipSuccess && device >= 0 && device < kMaxDevices) raised[device].store(true, std::memory_order_release);
  return e;
}

// Launches a kernel; `done` (may be null) is recorded by the kernel's own completion, which costs a small call 1.4 us
// less than an event recorded behind it (a packet of its own), and waiting for it 2.3 us less than a wait for the stream.
template <typename... Params, typename... Args>
hipError_t StartKernel(void (*kernel)(Params...), dim3 grid, dim3 block, size_t ldsBytes, hipStream_t stream, hipEvent_t done,
                       Args... args) {
  if (done) hipExtLaunchKernelGGL(kernel, grid, block, (uint32_t)ldsBytes, stream, nullptr, done, 0, static_cast<Params>(args)...);
  else kernel<<<grid, block, ldsBytes, stream>>>(static_cast<Params>(args)...);
  return hipGetLastError();
}

template <int K, int PF, int W, int V>
hipError_t LaunchWalkVariant(const WalkParams &p, dim3 grid, dim3 block, size_t ldsBytes, hipStream_t stream) {
  hipError_t e = AllowFullLds<&WalkRowsLdsKernel<K, PF, W, V>>();
  if (e != hipSuccess) return e;
  return StartKernel(&WalkRowsLdsKernel<K, PF, W, V>, grid, block, ldsBytes, stream, p.done, p.x, p.nodes16, p.bundles, p.bundleRoots,
                     p.groups, p.s, p.out, p.classOut, p.partial, p.leafIds, p.nodeOrigin, p.slotTree,
                     reinterpret_cast<const U32x2 *>(p.tailNodes), p.tailOrigin);
}

template <int K, int W, int V>
hipError_t LaunchSplitVariant(const WalkParams &p, dim3 block, size_t ldsBytes, hipStream_t stream) {
  hipError_t e = AllowFullLds<&WalkRowsSplitKernel<K, W, V>>();
  if (e != hipSuccess) return e;
  return StartKernel(&WalkRowsSplitKernel<K, W, V>, dim3((unsigned)p.splitBlocks), block, ldsBytes, stream, p.done, p.x, p.nodes16, p.bundles,
                     p.bundleRoots, p.groups, p.s, p.partial);
}

// The variants for where the last level's leaves are (rank tiles: always in LDS).
template <int K, int W, int V>
hipError_t LaunchSplitLeaves(const WalkParams &p, dim3 block, size_t ldsBytes, hipStream_t stream) {
  if constexpr (IsRankTile(W)) {
    return p.s.leavesOutside ? hipErrorInvalidValue : LaunchSplitVariant<K, W, V>(p, block, ldsBytes, stream);
  } else {
    return p.s.leavesOutside ? LaunchSplitVariant<K, W, V | kWalkOutside>(p, block, ldsBytes, stream)
                             : LaunchSplitVariant<K, W, V>(p, block, ldsBytes, stream);
  }
}

template <int K, int W>
hipError_t LaunchSplit(const WalkParams &p, dim3 block, size_t ldsBytes, hipStream_t stream) {
  const int64_t rowBlocks = (p.s.rows + p.s.rowsPerBlock - 1) / p.s.rowsPerBlock;
  if (p.splitBlocks < 1 || p.splitBlocks > rowBlocks * p.s.numGroups || !p.partial || p.leafIds || p.s.deferTails || p.s.fuseArgmax)
    return hipErrorInvalidValue;
  return p.s.ownClasses ? LaunchSplitLeaves<K, W, kWalkOwn>(p, block, ldsBytes, stream)
                        : LaunchSplitLeaves<K, W, kWalkPlain>(p, block, ldsBytes, stream);
}

template <int K, int PF, int W, int V>
hipError_t LaunchWalkLeaves(const WalkParams &p, dim3 grid, dim3 block, size_t ldsBytes, hipStream_t stream) {
  if constexpr (IsRankTile(W)) {
    return p.s.leavesOutside ? hipErrorInvalidValue : LaunchWalkVariant<K, PF, W, V>(p, grid, block, ldsBytes, stream);
  } else {
    return p.s.leavesOutside ? LaunchWalkVariant<K, PF, W, V | kWalkOutside>(p, grid, block, ldsBytes, stream)
                             : LaunchWalkVariant<K, PF, W, V>(p, grid, block, ldsBytes, stream);
  }
}

template <int K, int PF, int W>
hipError_t LaunchWalkKP(const WalkParams &p, dim3 grid, dim3 block, size_t ldsBytes, hipStream_t stream) {
  if (p.leafIds) { // (the dump kernel walks every bundle to its full depth and leaves the arg-max to the finalize kernel)
    if (p.s.fuseArgmax || (p.s.deferTails && W != kTileF32Bytes)) return hipErrorInvalidValue;
    return LaunchWalkVariant<K, PF, W, kWalkDump>(p, grid, block, ldsBytes, stream);
  }
  if (p.s.ownClasses)
    return p.s.fuseArgmax ? LaunchWalkLeaves<K, PF, W, kWalkOwnFuse>(p, grid, block, ldsBytes, stream)
                          : LaunchWalkLeaves<K, PF, W, kWalkOwn>(p, grid, block, ldsBytes, stream);
  if (p.s.fuseArgmax) return LaunchWalkLeaves<K, PF, W, kWalkFuse>(p, grid, block, ldsBytes, stream);
  // deferred tails are built for the f32 tile with byte offsets only (the packer makes stubs for no other plan)
  if (p.s.deferTails) {
    if (W != kTileF32Bytes || p.s.numClasses > 0 || p.s.leavesOutside) return hipErrorInvalidValue;
    return LaunchWalkVariant<K, PF, kTileF32Bytes, kWalkDefer>(p, grid, block, ldsBytes, stream);
  }
  return LaunchWalkLeaves<K, PF, W, kWalkPlain>(p, grid, block, ldsBytes, stream);
}

template <int K, int W>
hipError_t LaunchWalkK(const WalkParams &p, int prefetch, dim3 grid, dim3 block, size_t ldsBytes, hipStream_t stream) {
  if (p.splitBlocks) return LaunchSplit<K, W>(p, block, ldsBytes, stream);
  if (p.directStaging) return LaunchWalkKP<K, 0, W>(p, grid, block, ldsBytes, stream);
  if (prefetch <= 4) return LaunchWalkKP<K, 4, W>(p, grid, block, ldsBytes, stream);
  if (prefetch <= 8) return LaunchWalkKP<K, 8, W>(p, grid, block, ldsBytes, stream);
  if (prefetch <= 16) return LaunchWalkKP<K, 16, W>(p, grid, block, ldsBytes, stream);
  return hipErrorInvalidValue;
}

template <int W>
hipError_t LaunchWalkW(const WalkParams &p, int interleave, int prefetch, dim3 grid, dim3 block, size_t ldsBytes,
                       hipStream_t stream) {
  switch (interleave) {
  case 1: return LaunchWalkK<1, W>(p, prefetch, grid, block, ldsBytes, stream);
  case 2: return LaunchWalkK<2, W>(p, prefetch, grid, block, ldsBytes, stream);
  case 4: return LaunchWalkK<4, W>(p, prefetch, grid, block, ldsBytes, stream);
  case 8: return LaunchWalkK<8, W>(p, prefetch, grid, block, ldsBytes, stream);
  default: return hipErrorInvalidValue;
  }
}

} // namespace

namespace {
// Outputs the walk kernels dereference must be there: a fused epilogue writes p.out (or p.classOut), everything
// else goes through p.partial.
bool OutputsConsistent(const WalkParams &p) {
  if (p.splitBlocks) return true; // (LaunchSplit)
  if (p.s.fuseArgmax) return p.s.numClasses > 0 && p.s.treeSlices == 1 && (p.out || p.classOut);
  if (p.s.numClasses > 0 || p.s.treeSlices > 1) return p.partial != nullptr;
  return p.out != nullptr || p.partial != nullptr;
}
} // namespace

hipError_t LaunchWalkRowsLds(const WalkParams &p, int interleave, int tileMode, size_t ldsBytes, hipStream_t stream) {
  if (p.s.rows <= 0) return hipSuccess;
  if (!OutputsConsistent(p)) return hipErrorInvalidValue;
  const int RB = p.s.rowsPerBlock, TT = p.s.treeThreads;
  if (ldsBytes > 160 * 1024 || RB < 64 || (RB & (RB - 1)) || TT < 1 || RB * TT > 1024) return hipErrorInvalidValue;
  const int64_t blocks = (p.s.rows + RB - 1) / RB;
  if (blocks > 0x7FFFFFFF || p.s.treeSlices < 1 || p.s.treeSlices > 65535) return hipErrorInvalidValue;
  // registers that hold the next tree group while the current one is walked
  const int prefetch = (int)((p.s.groupRegionBytes / 16 + RB * TT - 1) / (RB * TT));
  dim3 grid((unsigned)blocks, (unsigned)p.s.treeSlices), block((unsigned)(RB * TT));
  switch (tileMode) {
  case kTileF32Bytes: return LaunchWalkW<kTileF32Bytes>(p, interleave, prefetch, grid, block, ldsBytes, stream);
  case kTileF32Words: return LaunchWalkW<kTileF32Words>(p, interleave, prefetch, grid, block, ldsBytes, stream);
  case kTileRankU8:
    if (RB != 64) return hipErrorInvalidValue;
    return LaunchWalkW<kTileRankU8>(p, interleave, prefetch, grid, block, ldsBytes, stream);
  case kTileRankU16: // (tree groups always go straight from global memory into LDS)
    if ((int64_t)((p.s.numFeatures + 2) / 2) * RB * 4 > 0x10000) return hipErrorInvalidValue; // byte offsets
    if (p.splitBlocks) return hipErrorInvalidValue; // (the plan search tries this form on full batches only)
    switch (interleave) {
    case 1: return LaunchWalkKP<1, 0, kTileRankU16>(p, grid, block, ldsBytes, stream);
    case 2: return LaunchWalkKP<2, 0, kTileRankU16>(p, grid, block, ldsBytes, stream);
    case 4: return LaunchWalkKP<4, 0, kTileRankU16>(p, grid, block, ldsBytes, stream);
    case 8: return LaunchWalkKP<8, 0, kTileRankU16>(p, grid, block, ldsBytes, stream);
    default: return hipErrorInvalidValue;
    }
  default: return hipErrorInvalidValue;
  }
}

namespace {
template <int T, int K, int V>
hipError_t LaunchTiledVariant(const WalkParams &p, dim3 grid, dim3 block, size_t ldsBytes, hipStream_t stream) {
  hipError_t e = AllowFullLds<&WalkRowsTiledKernel<T, K, V>>();
  if (e != hipSuccess) return e;
  return StartKernel(&WalkRowsTiledKernel<T, K, V>, grid, block, ldsBytes, stream, p.done, p.x, p.nodes16, p.bundles, p.groups, p.s, p.out,
                     p.classOut, p.partial, p.leafIds, p.nodeOrigin, p.slotTree);
}

template <int T, int K>
hipError_t LaunchTiledTK(const WalkParams &p, dim3 grid, dim3 block, size_t ldsBytes, hipStream_t stream) {
  if (p.leafIds) {
    if (p.s.fuseArgmax) return hipErrorInvalidValue;
    return LaunchTiledVariant<T, K, kWalkDump>(p, grid, block, ldsBytes, stream);
  }
  if (p.s.fuseArgmax) return LaunchTiledVariant<T, K, kWalkFuse>(p, grid, block, ldsBytes, stream);
  return LaunchTiledVariant<T, K, kWalkPlain>(p, grid, block, ldsBytes, stream);
}

template <int T>
hipError_t LaunchTiledT(const WalkParams &p, int interleave, dim3 grid, dim3 block, size_t ldsBytes, hipStream_t stream) {
  switch (interleave) {
  case 1: return LaunchTiledTK<T, 1>(p, grid, block, ldsBytes, stream);
  case 2: return LaunchTiledTK<T, 2>(p, grid, block, ldsBytes, stream);
  case 4: return LaunchTiledTK<T, 4>(p, grid, block, ldsBytes, stream);
  default: return hipErrorInvalidValue;
  }
}
} // namespace

hipError_t LaunchWalkRowsTiled(const WalkParams &p, int tileSize, int interleave, size_t ldsBytes, hipStream_t stream) {
  if (p.s.rows <= 0) return hipSuccess;
  if (!OutputsConsistent(p)) return hipErrorInvalidValue;
  const int RB = p.s.rowsPerBlock, TT = p.s.treeThreads;
  if (ldsBytes > 160 * 1024 || RB < 64 || (RB & (RB - 1)) || TT < 1 || RB * TT > 1024) return hipErrorInvalidValue;
  // feature offsets are byte offsets into the f32 row tile: the tile has to end below 64 KB
  if ((int64_t)(p.s.numFeatures + 1) * RB * 4 > 0x10000) return hipErrorInvalidValue;
  const int64_t blocks = (p.s.rows + RB - 1) / RB;
  if (blocks > 0x7FFFFFFF || p.s.treeSlices < 1 || p.s.treeSlices > 65535) return hipErrorInvalidValue;
  dim3 grid((unsigned)blocks, (unsigned)p.s.treeSlices), block((unsigned)(RB * TT));
  switch (tileSize) {
  case 2: return LaunchTiledT<2>(p, interleave, grid, block, ldsBytes, stream);
  case 3: return LaunchTiledT<3>(p, interleave, grid, block, ldsBytes, stream);
  case 4: return LaunchTiledT<4>(p, interleave, grid, block, ldsBytes, stream);
  case 5: case 6: case 7: case 8: // one eight-slot tile for all four; the packer fills as many slots as the tile size says
    return LaunchTiledT<kMaxTileSize>(p, interleave, grid, block, ldsBytes, stream);
  default: return hipErrorInvalidValue;
  }
}

namespace {
template <int K, int PF>
hipError_t LaunchTreeParallelKP(const WalkParams &p, dim3 grid, dim3 block, size_t ldsBytes, hipStream_t stream) {
  if (p.leafIds) {
    hipError_t e = AllowFullLds<&WalkTreeParallelKernel<K, PF, true>>();
    if (e != hipSuccess) return e;
    return StartKernel(&WalkTreeParallelKernel<K, PF, true>, grid, block, ldsBytes, stream, p.done, p.x, p.nodes16, p.bundles, p.groups, p.s,
                       p.out, p.partial, p.leafIds, p.nodeOrigin, p.slotTree);
  }
  hipError_t e = AllowFullLds<&WalkTreeParallelKernel<K, PF, false>>();
  if (e != hipSuccess) return e;
  return StartKernel(&WalkTreeParallelKernel<K, PF, false>, grid, block, ldsBytes, stream, p.done, p.x, p.nodes16, p.bundles, p.groups, p.s,
                     p.out, p.partial, nullptr, nullptr, nullptr);
}

template <int K>
hipError_t LaunchTreeParallelK(const WalkParams &p, int prefetch, dim3 grid, dim3 block, size_t ldsBytes,
                               hipStream_t stream) {
  if (prefetch <= 4) return LaunchTreeParallelKP<K, 4>(p, grid, block, ldsBytes, stream);
  if (prefetch <= 8) return LaunchTreeParallelKP<K, 8>(p, grid, block, ldsBytes, stream);
  if (prefetch <= 16) return LaunchTreeParallelKP<K, 16>(p, grid, block, ldsBytes, stream);
  return hipErrorInvalidValue;
}
} // namespace

hipError_t LaunchWalkTreeParallel(const WalkParams &p, int interleave, size_t ldsBytes, hipStream_t stream) {
  if (p.s.rows <= 0) return hipSuccess;
  if (ldsBytes > 160 * 1024 || p.s.rowsPerBlock < 1 || p.s.treeLanes < 1) return hipErrorInvalidValue;
  const int threads = p.s.rowsPerBlock * p.s.treeLanes;
  if (threads > 1024 || threads % 64 != 0) return hipErrorInvalidValue;
  const int64_t blocks = (p.s.rows + p.s.rowsPerBlock - 1) / p.s.rowsPerBlock;
  if (blocks > 0x7FFFFFFF || p.s.treeSlices < 1 || p.s.treeSlices > 65535) return hipErrorInvalidValue;
  const int prefetch = (int)((p.s.groupRegionBytes / 16 + threads - 1) / threads);
  dim3 grid((unsigned)blocks, (unsigned)p.s.treeSlices), block((unsigned)threads);
  switch (interleave) {
  case 1: return LaunchTreeParallelK<1>(p, prefetch, grid, block, ldsBytes, stream);
  case 2: return LaunchTreeParallelK<2>(p, prefetch, grid, block, ldsBytes, stream);
  case 4: return LaunchTreeParallelK<4>(p, prefetch, grid, block, ldsBytes, stream);
  case 8: return LaunchTreeParallelK<8>(p, prefetch, grid, block, ldsBytes, stream);
  default: return hipErrorInvalidValue;
  }
}

namespace {
template <int K>
hipError_t LaunchGlobalK(const WalkParams &p, dim3 grid, dim3 block, hipStream_t stream) {
  if (p.leafIds)
    return StartKernel(&WalkGlobalKernel<K, true>, grid, block, 0, stream, p.done, p.x, p.globalNodes, p.globalTrees, p.s, p.out, p.partial,
                       p.leafIds);
  return StartKernel(&WalkGlobalKernel<K, false>, grid, block, 0, stream, p.done, p.x, p.globalNodes, p.globalTrees, p.s, p.out, p.partial,
                     nullptr);
}
} // namespace

hipError_t LaunchWalkGlobal(const WalkParams &p, int interleave, hipStream_t stream) {
  if (p.s.rows <= 0) return hipSuccess;
  const int threads = p.s.rowsPerBlock;
  if (threads < 64 || threads > 1024 || threads % 64 != 0) return hipErrorInvalidValue;
  const int64_t blocks = (p.s.rows + threads - 1) / threads;
  if (blocks > 0x7FFFFFFF || p.s.treeSlices < 1 || p.s.treeSlices > 65535) return hipErrorInvalidValue;
  dim3 grid((unsigned)blocks, (unsigned)p.s.treeSlices), block((unsigned)threads);
  switch (interleave) {
  case 1: return LaunchGlobalK<1>(p, grid, block, stream);
  case 2: return LaunchGlobalK<2>(p, grid, block, stream);
  case 4: return LaunchGlobalK<4>(p, grid, block, stream);
  case 8: return LaunchGlobalK<8>(p, grid, block, stream);
  default: return hipErrorInvalidValue;
  }
}

hipError_t LaunchBinRows(const float *x, const float *table, uint8_t *ranks, int64_t rows, int numFeatures,
                         int tableDepth, int chunkFeatures, hipStream_t stream) {
  if (rows <= 0) return hipSuccess;
  if (chunkFeatures != kBinFeatures) return hipErrorInvalidValue;
  const size_t ldsBytes = (size_t)tableDepth * kBinFeatures * sizeof(float) + (size_t)kBinWaves * 64 * kBinLaneStride;
  if (ldsBytes > 160 * 1024) return hipErrorInvalidValue;
  const int64_t rowBlocks = (rows + kBinRows - 1) / kBinRows;
  const int chunks = (numFeatures + kBinFeatures - 1) / kBinFeatures;
  // enough blocks to fill the chip, each amortising its table load over several row blocks per wave
  int64_t perBlock = (rowBlocks * chunks + 2047) / 2048;
  if (perBlock < kBinWaves) perBlock = kBinWaves;
  if (perBlock > 64 * kBinWaves) perBlock = 64 * kBinWaves;
  const int64_t rowGroups = (rowBlocks + perBlock - 1) / perBlock;
  const int64_t blocks = (rowGroups + 7) / 8 * 8 * chunks; // row groups padded to the 8 XCDs
  if (blocks > 0x7FFFFFFF) return hipErrorInvalidValue;
  const dim3 grid((unsigned)blocks), block(kBinWaves * 64);
#define TBAMD_BIN_CASE(LEVELS)                                                                                         \
  case (1 << LEVELS) - 1: {                                                                                            \
    hipError_t e = AllowFullLds<&BinRowsKernel<LEVELS>>();                                                             \
    if (e != hipSuccess) return e;                                                                                     \
    BinRowsKernel<LEVELS><<<grid, block, ldsBytes, stream>>>(x, table, ranks, rows, numFeatures, (int)perBlock,       \
                                                             chunks);                                                  \
    return hipGetLastError();                                                                                          \
  }
  switch (tableDepth) {
    TBAMD_BIN_CASE(1)
    TBAMD_BIN_CASE(2)
    TBAMD_BIN_CASE(3)
    TBAMD_BIN_CASE(4)
    TBAMD_BIN_CASE(5)
    TBAMD_BIN_CASE(6)
    TBAMD_BIN_CASE(7)
    TBAMD_BIN_CASE(8)
  default: return hipErrorInvalidValue;
  }
#undef TBAMD_BIN_CASE
}

hipError_t LaunchRankRows16(const float *x, const float *tables, const RankFeatureDesc *features, const RankChunkDesc *chunks,
                            int numChunks, uint32_t maxChunkEntries, uint32_t maxChunkFeatures, uint16_t *ranks, int64_t rows,
                            int numFeatures, int rowsPerBlock, hipStream_t stream) {
  if (rows <= 0) return hipSuccess;
  const uint32_t tableRegionBytes = (maxChunkEntries * (uint32_t)sizeof(float) + 15u) & ~15u;
  const size_t ldsBytes = (size_t)tableRegionBytes + (size_t)maxChunkFeatures * kRankStride * sizeof(float);
  if (numChunks < 1 || ldsBytes > 160 * 1024 || rowsPerBlock < 64 || rowsPerBlock % 64 != 0) return hipErrorInvalidValue;
  const int64_t rowBlocks = (rows + rowsPerBlock - 1) / rowsPerBlock;
  // whole row blocks (the walk copies whole tiles), in tiles of 1024 rows: smaller row blocks are ranked up to the
  // next multiple of 1024 rows, which the rank buffer has to hold
  const int64_t rowTiles = (rowBlocks * rowsPerBlock + kRankTileRows - 1) / kRankTileRows;
  // enough blocks to fill the chip, each amortising its table load over a few thousand rows
  int64_t perBlock = (rowTiles * numChunks + 4095) / 4096;
  if (perBlock < 2) perBlock = 2;
  if (perBlock > 16) perBlock = 16;
  const int64_t ranges = (rowTiles + perBlock - 1) / perBlock;
  const int64_t blocks = (ranges + 7) / 8 * 8 * numChunks; // row ranges padded to the 8 XCDs
  if (blocks > 0x7FFFFFFF) return hipErrorInvalidValue;
  hipError_t e = AllowFullLds<&RankRows16Kernel>();
  if (e != hipSuccess) return e;
  RankRows16Kernel<<<dim3((unsigned)blocks), dim3(kRankWaves * 64), ldsBytes, stream>>>(
      x, tables, features, chunks, reinterpret_cast<uint32_t *>(ranks), rows, numFeatures, rowsPerBlock, numChunks, (int)perBlock,
      rowTiles, tableRegionBytes);
  return hipGetLastError();
}

hipError_t LaunchFewRows(const FewRowsParams &p, hipStream_t stream) {
  if (p.rows <= 0) return hipSuccess;
  const FewRowsShape s = ShapeOfFewRows(p.rows, p.numFeatures, p.numTrees, p.numClasses);
  if (p.numTrees < 1 || s.ldsBytes > kFewRowsLds) return hipErrorInvalidValue;
  if (p.numClasses == 0 ? !p.out : !(p.out || p.classOut || p.margins || p.probabilities)) return hipErrorInvalidValue;
  const int64_t blocks = (p.rows + s.rowsPerBlock - 1) / s.rowsPerBlock;
  return StartKernel(&FewRowsKernel, dim3((unsigned)blocks), dim3((unsigned)s.threads), s.ldsBytes, stream, p.done, p, s.rowsPerBlock,
                     (int)s.leafStride);
}

hipError_t LaunchRankStream(const RankStreamParams &p, hipStream_t stream) {
  if (p.rows <= 0) return hipSuccess;
  const int waves = StreamWaves(p.numFeatures);
  if (waves < 1 || p.numFeatures > kStreamMaxFeatures || p.numBundles < 1 || (p.chains != 2 && p.chains != 4) || p.slices < 1 || p.slices > 65535) return hipErrorInvalidValue;
  if (p.slices > 1 ? !p.partial : !p.out) return hipErrorInvalidValue;
  const int64_t blocks = ((p.rows + kStreamRows - 1) / kStreamRows + 15) / 16 * 16;
  const size_t ldsBytes = (((size_t)(p.numFeatures + 1) * kStreamRows + 15) & ~(size_t)15) + (size_t)waves * 2 * kStreamBundleBytes;
  if (blocks > 0x7FFFFFFF || ldsBytes > 160 * 1024) return hipErrorInvalidValue;
  if ((int64_t)p.numFeatures * 2 > (int64_t)waves * 64 * kStreamTilePieces) return hipErrorInvalidValue;
  // (a workgroup has a compute unit's LDS to itself and goes on with other rows; multiples of 16 keep the XCDs' row blocks)
  const int64_t groups = std::min<int64_t>(blocks, std::max(16, p.computeUnits / 16 * 16));
  const dim3 grid((unsigned)groups, (unsigned)p.slices), block((unsigned)waves * 64);
  const bool stays = groups < blocks, four = p.chains == 4;
  hipError_t e = stays ? (four ? AllowFullLds<&RankStreamKernel<4, true>>() : AllowFullLds<&RankStreamKernel<2, true>>())
                       : (four ? AllowFullLds<&RankStreamKernel<4, false>>() : AllowFullLds<&RankStreamKernel<2, false>>());
  if (e != hipSuccess) return e;
  return StartKernel(stays ? (four ? &RankStreamKernel<4, true> : &RankStreamKernel<2, true>)
                           : (four ? &RankStreamKernel<4, false> : &RankStreamKernel<2, false>),
                     grid, block, ldsBytes, stream, p.done, p.ranks, p.words, p.values, p.bundles, p.rows, p.numFeatures, p.numBundles, p.slices, p.transform, p.initialValue,
                     p.slices > 1 ? nullptr : p.out, p.slices > 1 ? p.partial : nullptr);
}

hipError_t LaunchFinalize(const FinalizeParams &p, hipStream_t stream) {
  if (p.rows <= 0) return hipSuccess;
  if (p.numClasses > 0) {
    // A sum per lane, and 8 rows at least; about rows / 1024 of a batch that has more than 1024 such blocks: the chip is full then,
    // and a block in which few lanes finish a row costs more than the wait of one that takes several sums a lane.  (As many as make
    // whole rounds of the lanes: 30 rows instead of 28 of nine classes took 31377 rows 0.8 us longer.)  Calls with sums and softmax
    // of 40 trees, a sum per lane, 64, 128 and 256 rows: 5 classes 65537 rows 24.7, 24.8, 25.0 and 25.3 us, 150000 34.0, 33.7, 32.3,
    // 31.0, 700000 75.4, 74.1, 68.7, 67.1; 12 classes 25000 rows 23.8, 24.3, 25.9, 27.6, 65537 30.5, 28.6, 30.3, 31.0, 300000 67.4,
    // 58.2, 58.5, 57.2; 16 classes 700000 rows 152.5, 120.6, 118.9 and (240 rows) 126.0.
    const int64_t stride = p.numClasses | 1, perLane = std::max(8, 256 / p.numClasses);
    const int64_t most = std::max<int64_t>(perLane, std::min<int64_t>(256, kFinalizeLds / 2 / stride));
    const int64_t wanted = std::max<int64_t>(1, (p.rows / 1024 + perLane / 2) / perLane) * perLane;
    const int64_t perBlock = std::min<int64_t>(kFinalizeLds / stride, std::min(most, wanted));
    const int64_t blocks = (p.rows + perBlock - 1) / perBlock;
    const size_t sumBytes = (size_t)perBlock * (size_t)(p.numClasses | 1) * sizeof(double), rowBytes = (size_t)perBlock * 2 * sizeof(double);
    if (blocks > 0x7FFFFFFF) return hipErrorInvalidValue;
    if (sumBytes + rowBytes > 64 * 1024)
      return StartKernel(&FinalizeManyClassesKernel, dim3((unsigned)((p.rows + 255) / 256)), dim3(256), 0, stream, p.done, p);
    const int groups = p.treeSlices >= kClassPartsShared && sumBytes * 2 + rowBytes <= 64 * 1024 ? 2 : 1;
    return StartKernel(&FinalizeClassesKernel, dim3((unsigned)blocks), dim3((unsigned)(256 * groups)), sumBytes * groups + rowBytes, stream,
                       p.done, p, (int)perBlock);
  }
  if (p.treeSlices >= kWideFinalizeSlices && p.rows <= kWideFinalizeRows)
    return StartKernel(p.treeSlices < 8 ? &FinalizeWideKernel<4> : &FinalizeWideKernel<8>, dim3((unsigned)((p.rows + 63) / 64)),
                       dim3(p.treeSlices < 8 ? 256 : 512), 0, stream, p.done, p);
  const int64_t blocks = (p.rows + 255) / 256;
  return StartKernel(&FinalizeKernel, dim3((unsigned)blocks), dim3(256), 0, stream, p.done, p);
}

} // namespace tbamd
