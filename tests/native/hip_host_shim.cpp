// Host-only stand-in for the HIP runtime and for the kernel launchers of kernels.h, so that the runner
// and the C ABI (runner.cpp, runtime.cpp) can run under AddressSanitizer / ThreadSanitizer without a GPU.
//
// "Device" memory is ordinary heap memory, so every buffer the library allocates gets the sanitizer's
// red zones; copies are memcpy; streams and events are tokens.  The launchers below interpret the packed
// model on the CPU with the kernels' addressing rules (group-relative node addresses, pre-multiplied
// feature offsets, rank tiles, per-class partial sums, tree slices, finalize), reading every input and
// writing every output element the kernels touch: a buffer sized or indexed wrongly by the host code is
// reported by the sanitizer, and a wrongly packed model gives wrong predictions.  An asynchronous copy happens no sooner
// than its stream is waited for or has something behind it, so a buffer that is given up too early shows; a wait for an event
// that nothing has recorded since the last wait ends the run.  Test infrastructure only.
#include "kernels.h"

#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <vector>

namespace {
std::mutex gMutex;
std::map<const void *, std::pair<size_t, bool>> gAllocations; // pointer -> (bytes, pinned host)
hipError_t gLastError = hipSuccess;

struct Copy {
  void *dst;
  const void *src;
  size_t bytes;
};
struct Stream {
  long queued = 0, waited = 0; // pieces of work handed over, and how many of them the host has waited for
  std::vector<Copy> copies;    // still to be done
};
std::map<hipStream_t, Stream> gStreams;
struct Event {
  bool recorded = false; // ... and not waited for since
  hipStream_t stream = nullptr;
  long at = 0;
};
Event &EventOf(hipEvent_t event) { return *reinterpret_cast<Event *>(event); }

// (with gMutex held)
void DoCopies(Stream &stream) {
  for (const Copy &c : stream.copies)
    if (c.bytes) std::memcpy(c.dst, c.src, c.bytes);
  stream.copies.clear();
}

hipError_t Fail(hipError_t e) {
  gLastError = e;
  return e;
}
} // namespace

extern "C" {

hipError_t hipMalloc(void **ptr, size_t size) {
  if (!ptr) return Fail(hipErrorInvalidValue);
  *ptr = std::malloc(size ? size : 1);
  if (!*ptr) return Fail(hipErrorOutOfMemory);
  std::memset(*ptr, 0xA5, size); // device memory starts with garbage
  std::lock_guard<std::mutex> lock(gMutex);
  gAllocations[*ptr] = {size, false};
  return hipSuccess;
}

hipError_t hipFree(void *ptr) {
  if (!ptr) return hipSuccess;
  {
    std::lock_guard<std::mutex> lock(gMutex);
    for (auto &stream : gStreams) DoCopies(stream.second); // (the runtime waits too)
    if (!gAllocations.erase(ptr)) return Fail(hipErrorInvalidValue);
  }
  std::free(ptr);
  return hipSuccess;
}

hipError_t hipHostMalloc(void **ptr, size_t size, unsigned int) {
  if (!ptr) return Fail(hipErrorInvalidValue);
  *ptr = std::malloc(size ? size : 1);
  if (!*ptr) return Fail(hipErrorOutOfMemory);
  std::lock_guard<std::mutex> lock(gMutex);
  gAllocations[*ptr] = {size, true};
  return hipSuccess;
}

hipError_t hipHostFree(void *ptr) { return hipFree(ptr); }

hipError_t hipMemcpy(void *dst, const void *src, size_t bytes, hipMemcpyKind) {
  if (bytes) std::memcpy(dst, src, bytes);
  return hipSuccess;
}

hipError_t hipMemcpyAsync(void *dst, const void *src, size_t bytes, hipMemcpyKind, hipStream_t stream) {
  std::lock_guard<std::mutex> lock(gMutex);
  ++gStreams[stream].queued;
  gStreams[stream].copies.push_back(Copy{dst, src, bytes});
  return hipSuccess;
}

hipError_t hipPointerGetAttributes(hipPointerAttribute_t *attr, const void *ptr) {
  std::lock_guard<std::mutex> lock(gMutex);
  auto it = gAllocations.upper_bound(ptr);
  if (it == gAllocations.begin()) return Fail(hipErrorInvalidValue);
  --it;
  const char *base = static_cast<const char *>(it->first);
  if (static_cast<const char *>(ptr) >= base + it->second.first) return Fail(hipErrorInvalidValue);
  std::memset(attr, 0, sizeof(*attr));
  attr->type = it->second.second ? hipMemoryTypeHost : hipMemoryTypeDevice;
  return hipSuccess;
}

hipError_t hipStreamCreateWithFlags(hipStream_t *stream, unsigned int) {
  *stream = reinterpret_cast<hipStream_t>(new int(0));
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t stream) {
  {
    std::lock_guard<std::mutex> lock(gMutex);
    DoCopies(gStreams[stream]);
    gStreams.erase(stream);
  }
  delete reinterpret_cast<int *>(stream);
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t stream) {
  std::lock_guard<std::mutex> lock(gMutex);
  Stream &s = gStreams[stream];
  DoCopies(s);
  s.waited = s.queued;
  return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t event, unsigned int) {
  if (!EventOf(event).recorded) std::abort(); // orders nothing
  return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t *event) {
  *event = reinterpret_cast<hipEvent_t>(new Event);
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t *event, unsigned) { return hipEventCreate(event); }
hipError_t hipEventDestroy(hipEvent_t event) {
  delete &EventOf(event);
  return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t event, hipStream_t stream) {
  std::lock_guard<std::mutex> lock(gMutex);
  DoCopies(gStreams[stream]);
  EventOf(event) = Event{true, stream, gStreams[stream].queued};
  return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t event) {
  std::lock_guard<std::mutex> lock(gMutex);
  Event &e = EventOf(event);
  if (!e.recorded) std::abort(); // waits for nothing
  e.recorded = false;
  const auto stream = gStreams.find(e.stream);
  if (stream != gStreams.end()) stream->second.waited = std::max(stream->second.waited, e.at);
  return hipSuccess;
}
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) {
  static float fake = 1.0f; // every measurement a little longer than the last: plan searches keep the first
  fake += 0.001f;
  *ms = fake;
  return hipSuccess;
}
hipError_t hipGetDeviceCount(int *count) {
  *count = 1;
  return hipSuccess;
}
hipError_t hipGetDevice(int *device) {
  *device = 0;
  return hipSuccess;
}
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *prop, int) {
  std::memset(prop, 0, sizeof(*prop));
  const char *units = std::getenv("SHIM_COMPUTE_UNITS"); // (few of them: small batches already run in several rounds of blocks)
  prop->multiProcessorCount = units ? std::atoi(units) : 256;
  prop->sharedMemPerBlock = 160 * 1024;
  return hipSuccess;
}
hipError_t hipGetSymbolAddress(void **devPtr, const void *symbol) {
  *devPtr = const_cast<void *>(symbol);
  return hipSuccess;
}
const char *hipGetErrorString(hipError_t e) { return e == hipSuccess ? "no error" : "emulated HIP error"; }
hipError_t hipGetLastError(void) {
  const hipError_t e = gLastError;
  gLastError = hipSuccess;
  return e;
}

// Streams with work that nobody has waited for, the default stream and `except` left out.
int shimBusyStreams(hipStream_t except) {
  std::lock_guard<std::mutex> lock(gMutex);
  int busy = 0;
  for (const auto &stream : gStreams) busy += stream.first && stream.first != except && stream.second.waited < stream.second.queued;
  return busy;
}
long shimLaunchesToGo = -1; // launches until one fails (negative: none does)
long shimNoLaunches = 0;    // every launch fails
long shimFewRows = 0, shimSplits = 0, shimStreams = 0, shimDeferred = 0; // launches of the forms that stand beside the launch plans' kernels

} // extern "C"

namespace tbamd {

namespace {

uint32_t Bits(float v) {
  uint32_t u;
  std::memcpy(&u, &v, sizeof(u));
  return u;
}

// A kernel starts behind its stream's copies ...
bool Refused(hipStream_t stream) {
  std::lock_guard<std::mutex> lock(gMutex);
  if (shimLaunchesToGo >= 0 && shimLaunchesToGo-- == 0) return true;
  if (shimNoLaunches) return true;
  DoCopies(gStreams[stream]);
  ++gStreams[stream].queued;
  return false;
}
// ... and records its parameters' event when it is done.
hipError_t Launched(hipEvent_t done, hipStream_t stream) { return done ? hipEventRecord(done, stream) : hipSuccess; }

// One row through groups [gBegin, gEnd) of an LDS-layout model.  `stride` is the node-offset distance between
// two features; rankRows: x points at the rank tile [row block][feature][64 rows].
// rankRows: 0 f32 rows, 1 one-byte ranks, 2 two-byte ranks ([row block][feature pair][row][2], `stride` = bytes of
// one feature pair's column = rows per block x 4)
void WalkRowLds(const WalkParams &p, int K, uint32_t stride, int rankRows, int64_t row, int gBegin, int gEnd, double *classSums,
                bool *classSeen, bool leavesOutside) {
  const DeviceNode *nodes = reinterpret_cast<const DeviceNode *>(p.nodes16);
  const int F = p.s.numFeatures;
  for (int g = gBegin; g < gEnd; ++g) {
    const DeviceGroup grp = p.groups[g];
    for (uint32_t b = 0; b < grp.bundleCount; ++b) {
      const DeviceBundle bd = p.bundles[grp.bundleBegin + b];
      for (int k = 0; k < K; ++k) {
        uint32_t addr = bd.root[k];
        for (uint32_t d = 0; d < bd.depth; ++d) {
          if (addr % kNodeBytes != 0 || addr / kNodeBytes >= grp.nodeCount) std::abort(); // pointer outside the group
          const DeviceNode node = nodes[grp.nodeBegin + addr / kNodeBytes];
          const uint32_t offset = MetaFeature(node.meta);
          const uint32_t f = rankRows == 2 ? offset / stride * 2u + ((offset >> 1) & 1u) : offset / stride;
          if ((rankRows == 2 ? (offset % stride) & ~2u : offset % stride) != 0 || (int)f > F) std::abort(); // offset outside the row tile
          bool left;
          if (rankRows == 2) {
            const uint16_t *ranks = reinterpret_cast<const uint16_t *>(p.x);
            const int64_t RB = stride / 4, pairs = (F + 2) / 2;
            const uint32_t rank = ranks[(((row / RB) * pairs + f / 2) * RB + row % RB) * 2 + (f & 1)]; // (the pad feature's slot holds 0)
            left = rank <= Bits(node.value);
          } else if (rankRows) {
            const uint8_t *ranks = reinterpret_cast<const uint8_t *>(p.x);
            const uint32_t rank = (int)f == F ? 0u : ranks[((row / 64) * F + f) * 64 + (row % 64)];
            left = rank <= Bits(node.value);
          } else {
            const float x = (int)f >= F ? -INFINITY : p.x[row * F + f]; // (the pad feature and the stub feature hold -inf)
            left = x < node.value;
          }
          addr = MetaChild(node.meta) + (left ? 0u : leavesOutside && d + 1 == bd.depth ? 4u : kNodeBytes); // (the last level: leaves of 4 bytes)
        }
        if (addr % 4 != 0 || (addr < grp.nodeCount * kNodeBytes ? addr % kNodeBytes != 0 : !leavesOutside || addr / kNodeBytes >= grp.imageCount)) std::abort();
        float leafValue; // (of the group's image, in LDS or not)
        std::memcpy(&leafValue, reinterpret_cast<const char *>(nodes + grp.nodeBegin) + addr, sizeof(leafValue));
        bool inTail = false;
        uint32_t at = 0;
        if (p.s.deferTails) {
          // a stub (NaN value, child pointer one node before itself) stands for the node of the tail array its
          // payload names: the walk goes on there for at most tailDepth steps
          const DeviceNode stop = nodes[grp.nodeBegin + addr / kNodeBytes];
          if (rankRows != 0 || stride == 0) std::abort();
          if (stop.value != stop.value) { // a NaN marks a stub; its payload is the tail index
            if (!bd.hasStubs || MetaChild(stop.meta) + kNodeBytes != addr || (Bits(stop.value) & ~kStubIndexMask) != kStubValueBits ||
                !p.tailNodes || (p.leafIds && !p.tailOrigin))
              std::abort();
            inTail = true;
            at = Bits(stop.value) & kStubIndexMask;
            if (at == 0) std::abort();
            for (int d = 0; d < p.s.tailDepth; ++d) {
              const DeviceNode node = p.tailNodes[at];
              const uint32_t f = node.meta & ((1u << kTailFeatureBits) - 1u);
              if ((int)f > F) std::abort();
              const float x = (int)f == F ? -INFINITY : p.x[row * F + f];
              at = (node.meta >> kTailFeatureBits) + (x < node.value ? 0u : 1u);
            }
            const DeviceNode leaf = p.tailNodes[at];
            if ((leaf.meta >> kTailFeatureBits) != at || (leaf.meta & ((1u << kTailFeatureBits) - 1u)) != (uint32_t)F) std::abort(); // tailDepth must reach a leaf
          }
        }
        if (inTail) {
          classSums[0] += (double)p.tailNodes[at].value;
          classSeen[0] = true;
          if (p.leafIds) {
            const int tree = p.slotTree[bd.firstSlot + k];
            if (tree >= 0) p.leafIds[row * p.s.numTrees + tree] = p.tailOrigin[at];
          }
          continue;
        }
        const int cls = p.s.numClasses > 0 ? (int)bd.classId : 0;
        if (p.s.numClasses > 0 && cls >= p.s.numClasses) { // a tree thread without a class: bundles without trees, no sum
          if (!p.s.ownClasses || cls >= p.s.treeThreads || leafValue != 0.0f) std::abort();
          if (p.leafIds && p.slotTree[bd.firstSlot + k] >= 0) std::abort();
          continue;
        }
        classSums[cls] += (double)leafValue;
        classSeen[cls] = true;
        if (p.leafIds) {
          const int tree = p.slotTree[bd.firstSlot + k];
          if (tree >= 0) p.leafIds[row * p.s.numTrees + tree] = p.nodeOrigin[grp.nodeBegin * 2 + addr / 4];
        }
      }
    }
  }
}

void StoreRow(const WalkParams &p, int64_t row, int slice, const double *classSums) {
  const int C = p.s.numClasses;
  if (p.s.fuseArgmax) { // the kernel's own running arg-max (ties go to the larger class id)
    if (C <= 0 || p.s.treeSlices != 1 || p.partial || (!p.out && !p.classOut)) std::abort();
    float best = -INFINITY;
    int bestClass = 0;
    for (int c = 0; c < C; ++c) {
      const float m = (float)(p.s.initialValue + classSums[c]);
      if (!(best > m)) best = m, bestClass = c;
    }
    if (p.classOut) p.classOut[row] = (int8_t)bestClass;
    else p.out[row] = (float)bestClass;
    return;
  }
  if (C > 0 || p.partial) {
    if (!p.partial) std::abort(); // classifiers always go through the finalize kernel
    double *dst = p.partial + ((int64_t)slice * p.s.rows + row) * (C > 0 ? C : 1);
    for (int c = 0; c < (C > 0 ? C : 1); ++c) dst[c] = classSums[c];
  } else {
    const double margin = p.s.initialValue + classSums[0];
    p.out[row] = (float)(p.s.transform == 1 ? 1.0 / (1.0 + std::exp(-margin)) : margin);
  }
}

// The walk's slots of the partial sums hold nothing yet: all of them can be written, and a part the walk leaves out shows.
void ClearPartial(const WalkParams &p, int64_t slots) {
  if (p.partial) std::fill_n(p.partial, slots * p.s.rows * std::max(1, p.s.numClasses), std::nan(""));
}

// leavesOutside: the last level of a bundle's walk is leaves of 4 bytes, not in LDS
hipError_t WalkLds(const WalkParams &p, int K, uint32_t stride, int rankRows, bool leavesOutside, hipStream_t stream) {
  if (K != 1 && K != 2 && K != 4 && K != 8) return hipErrorInvalidValue;
  if (p.s.treeSlices > 1 && !p.partial) std::abort(); // slices meet in the partial-sum buffer
  const int Cn = p.s.numClasses > 0 ? p.s.numClasses : 1;
  std::vector<double> sums((size_t)Cn);
  std::vector<char> seen((size_t)Cn);
  const auto walk = [&](int64_t firstRow, int64_t lastRow, int gBegin, int gEnd, int slot) {
    for (int64_t row = firstRow; row < lastRow; ++row) {
      std::fill(sums.begin(), sums.end(), 0.0);
      WalkRowLds(p, K, stride, rankRows, row, gBegin, gEnd, sums.data(), reinterpret_cast<bool *>(seen.data()), leavesOutside);
      StoreRow(p, row, slot, sums.data());
    }
  };
  if (p.splitBlocks) { // parts of the line of row blocks x groups, each in a slot of its row block
    const int64_t rowBlocks = (p.s.rows + p.s.rowsPerBlock - 1) / p.s.rowsPerBlock;
    if (p.splitBlocks < 1 || p.splitBlocks > rowBlocks * p.s.numGroups || !p.partial || p.leafIds || p.s.deferTails || p.s.fuseArgmax)
      return hipErrorInvalidValue;
    ++shimSplits;
    const SplitLine line{rowBlocks * p.s.numGroups, p.s.numGroups, p.splitBlocks};
    const int64_t slots = SplitLine::Slots(p.splitBlocks, rowBlocks);
    ClearPartial(p, slots);
    for (int64_t block = 0; block < p.splitBlocks; ++block)
      for (int64_t unit = line.FirstUnit(block), end = line.FirstUnit(block + 1); unit < end;) {
        const int64_t rowBlock = unit / line.groups, first = rowBlock * p.s.rowsPerBlock, slot = block - line.FirstBlock(rowBlock);
        const int gBegin = (int)(unit - rowBlock * line.groups), gEnd = (int)std::min<int64_t>(end - rowBlock * line.groups, line.groups);
        if (slot < 0 || slot >= slots || slot >= line.Parts(rowBlock)) std::abort();
        walk(first, std::min(p.s.rows, first + p.s.rowsPerBlock), gBegin, gEnd, (int)slot);
        unit += gEnd - gBegin;
      }
    return Launched(p.done, stream);
  }
  ClearPartial(p, p.s.treeSlices);
  for (int slice = 0; slice < p.s.treeSlices; ++slice)
    walk(0, p.s.rows, (int)(((int64_t)p.s.numGroups * slice) / p.s.treeSlices), (int)(((int64_t)p.s.numGroups * (slice + 1)) / p.s.treeSlices), slice);
  return Launched(p.done, stream);
}

} // namespace

hipError_t LaunchWalkRowsLds(const WalkParams &p, int interleave, int tileMode, size_t ldsBytes, hipStream_t stream) {
  if (p.s.rows <= 0) return hipSuccess;
  if (Refused(stream)) return hipErrorLaunchFailure;
  const int RB = p.s.rowsPerBlock, TT = p.s.treeThreads;
  if (ldsBytes > 160 * 1024 || RB < 64 || (RB & (RB - 1)) || TT < 1 || RB * TT > 1024) return hipErrorInvalidValue;
  if (p.s.treeSlices < 1 || p.s.treeSlices > 65535) return hipErrorInvalidValue;
  const int prefetch = (int)((p.s.groupRegionBytes / 16 + RB * TT - 1) / (RB * TT));
  if (prefetch > 16) return hipErrorInvalidValue;
  if (tileMode == 2 && RB != 64) return hipErrorInvalidValue;
  if (p.s.deferTails) ++shimDeferred;
  if (tileMode < 0 || tileMode > 3 || (tileMode == 3 && p.splitBlocks)) return hipErrorInvalidValue;
  if (tileMode == 3 && (int64_t)((p.s.numFeatures + 2) / 2) * RB * 4 > 0x10000) return hipErrorInvalidValue;
  if (tileMode >= 2 && p.s.leavesOutside && !p.leafIds) return hipErrorInvalidValue; // (rank tiles: always in LDS)
  const uint32_t stride = tileMode == 0 || tileMode == 3 ? (uint32_t)RB * 4u : tileMode == 1 ? (uint32_t)RB : (uint32_t)RB / 4u;
  return WalkLds(p, interleave, stride, tileMode == 3 ? 2 : tileMode == 2 ? 1 : 0, p.s.leavesOutside != 0, stream);
}

namespace {

// One tile step of the tiled layout (device_model.h): returns the byte address of the child tile.
uint32_t TileStepHost(const unsigned char *group, uint32_t groupBytes, uint32_t addr, int T, const float *row, int F,
                      uint32_t stride, int hops) {
  const uint32_t bytes = TileBytes(T);
  if (addr % 8 != 0 || addr + bytes > groupBytes) std::abort(); // tile outside the group
  const unsigned char *tile = group + addr;
  if (T > kMaxSelectTile) { // the eight-slot tile: { thr[8]; off[8]; links; childBase }
    float thr8[8];
    uint16_t off8[8], base;
    uint64_t links;
    std::memcpy(thr8, tile, 32);
    std::memcpy(off8, tile + 32, 16);
    std::memcpy(&links, tile + 48, 8);
    std::memcpy(&base, tile + 56, 2);
    uint32_t slot = 0;
    for (int hop = 0; hop < hops; ++hop) { // (the kernel follows `hops` links: they must reach a child)
      if (off8[slot] % stride != 0 || (int)(off8[slot] / stride) > F) std::abort();
      const int f = (int)(off8[slot] / stride);
      const float x = f == F ? -INFINITY : row[f];
      const uint32_t link = (uint32_t)(links >> (4 * slot + (x < thr8[slot] ? 32 : 0))) & 15u;
      if (link >= kTileLinkExit) return base + (link - kTileLinkExit) * bytes;
      slot = link + 1;
    }
    std::abort(); // links that never reach a child
  }
  float thr[kMaxTileSize];
  uint16_t off[kMaxTileSize], childBase;
  std::memcpy(thr, tile, (size_t)T * 4);
  std::memcpy(off, tile + T * 4, (size_t)T * 2);
  std::memcpy(&childBase, tile + T * 6, 2);
  uint64_t select = 0;
  if (T == 4) {
    uint16_t low;
    uint32_t high;
    std::memcpy(&low, tile + 26, 2);
    std::memcpy(&high, tile + 28, 4);
    select = (uint64_t)low | ((uint64_t)high << 16);
  } else {
    uint16_t s16;
    std::memcpy(&s16, tile + T * 6 + 2, 2);
    select = s16;
  }
  uint32_t outcome = 0;
  for (int i = 0; i < T; ++i) {
    if (off[i] % stride != 0 || (int)(off[i] / stride) > F) std::abort();
    const int f = (int)(off[i] / stride);
    const float x = f == F ? -INFINITY : row[f];
    outcome |= (x < thr[i] ? 1u : 0u) << i;
  }
  const uint32_t width = TileSelectBits(T);
  const uint32_t child = (uint32_t)(select >> (outcome * width)) & ((1u << width) - 1u);
  return childBase + child * bytes;
}

} // namespace

hipError_t LaunchWalkRowsTiled(const WalkParams &p, int tileSize, int interleave, size_t ldsBytes, hipStream_t stream) {
  if (p.s.rows <= 0) return hipSuccess;
  if (Refused(stream)) return hipErrorLaunchFailure;
  const int RB = p.s.rowsPerBlock, TT = p.s.treeThreads, T = tileSize, K = interleave;
  if (ldsBytes > 160 * 1024 || RB < 64 || (RB & (RB - 1)) || TT < 1 || RB * TT > 1024) return hipErrorInvalidValue;
  if ((int64_t)(p.s.numFeatures + 1) * RB * 4 > 0x10000) return hipErrorInvalidValue;
  if (p.s.treeSlices < 1 || p.s.treeSlices > 65535) return hipErrorInvalidValue;
  if (T < 2 || T > kMaxTileSize || (K != 1 && K != 2 && K != 4)) return hipErrorInvalidValue;
  if (p.s.treeSlices > 1 && !p.partial) std::abort();
  ClearPartial(p, p.s.treeSlices);
  const DeviceNode *nodes = reinterpret_cast<const DeviceNode *>(p.nodes16);
  const int F = p.s.numFeatures;
  const int Cn = p.s.numClasses > 0 ? p.s.numClasses : 1;
  std::vector<double> sums((size_t)Cn);
  for (int slice = 0; slice < p.s.treeSlices; ++slice) {
    const int gBegin = (int)(((int64_t)p.s.numGroups * slice) / p.s.treeSlices);
    const int gEnd = (int)(((int64_t)p.s.numGroups * (slice + 1)) / p.s.treeSlices);
    for (int64_t row = 0; row < p.s.rows; ++row) {
      std::fill(sums.begin(), sums.end(), 0.0);
      for (int g = gBegin; g < gEnd; ++g) {
        const DeviceGroup grp = p.groups[g];
        const unsigned char *group = reinterpret_cast<const unsigned char *>(nodes + grp.nodeBegin);
        for (uint32_t b = 0; b < grp.bundleCount; ++b) {
          const DeviceBundle bd = p.bundles[grp.bundleBegin + b];
          if (bd.peelDepth > bd.depth) std::abort();
          for (int k = 0; k < K; ++k) {
            uint32_t addr = bd.root[k];
            // the kernel stops early only when no lane moves any more, which leaves every lane where `depth`
            // steps would: the full walk is the specification
            for (uint32_t d = 0; d < bd.depth; ++d)
              addr = TileStepHost(group, grp.nodeCount * kNodeBytes, addr, T, p.x + row * F, F, (uint32_t)RB * 4u, p.s.tileHops);
            const uint32_t settled = TileStepHost(group, grp.nodeCount * kNodeBytes, addr, T, p.x + row * F, F, (uint32_t)RB * 4u, p.s.tileHops);
            if (settled != addr) std::abort(); // `depth` steps must end on a leaf tile
            float value;
            std::memcpy(&value, group + addr, 4);
            sums[p.s.numClasses > 0 ? bd.classId : 0] += (double)value;
            if (p.leafIds) {
              const int tree = p.slotTree[bd.firstSlot + k];
              if (tree >= 0) p.leafIds[row * p.s.numTrees + tree] = p.nodeOrigin[grp.nodeBegin * 2 + addr / 4];
            }
          }
        }
      }
      StoreRow(p, row, slice, sums.data());
    }
  }
  return Launched(p.done, stream);
}

hipError_t LaunchWalkTreeParallel(const WalkParams &p, int interleave, size_t ldsBytes, hipStream_t stream) {
  if (p.s.rows <= 0) return hipSuccess;
  if (Refused(stream)) return hipErrorLaunchFailure;
  if (ldsBytes > 160 * 1024 || p.s.rowsPerBlock < 1 || p.s.treeLanes < 1) return hipErrorInvalidValue;
  const int threads = p.s.rowsPerBlock * p.s.treeLanes;
  if (threads > 1024 || threads % 64 != 0) return hipErrorInvalidValue;
  if (p.s.treeSlices < 1 || p.s.treeSlices > 65535) return hipErrorInvalidValue;
  if ((int)((p.s.groupRegionBytes / 16 + threads - 1) / threads) > 16) return hipErrorInvalidValue;
  return WalkLds(p, interleave, 4u, 0, false, stream);
}

hipError_t LaunchWalkGlobal(const WalkParams &p, int interleave, hipStream_t stream) {
  if (p.s.rows <= 0) return hipSuccess;
  if (Refused(stream)) return hipErrorLaunchFailure;
  const int threads = p.s.rowsPerBlock;
  if (threads < 64 || threads > 1024 || threads % 64 != 0) return hipErrorInvalidValue;
  if (interleave != 1 && interleave != 2 && interleave != 4 && interleave != 8) return hipErrorInvalidValue;
  const int Cn = p.s.numClasses > 0 ? p.s.numClasses : 1;
  std::vector<double> sums((size_t)Cn);
  for (int slice = 0; slice < p.s.treeSlices; ++slice) {
    const int tBegin = (int)(((int64_t)p.s.numTrees * slice) / p.s.treeSlices);
    const int tEnd = (int)(((int64_t)p.s.numTrees * (slice + 1)) / p.s.treeSlices);
    for (int64_t row = 0; row < p.s.rows; ++row) {
      std::fill(sums.begin(), sums.end(), 0.0);
      for (int t = tBegin; t < tEnd; ++t) {
        const DeviceGlobalTree tree = p.globalTrees[t];
        uint32_t n = tree.root;
        for (uint32_t d = 0; d < tree.depth; ++d) {
          const DeviceGlobalNode node = p.globalNodes[n];
          if (node.feature != kGlobalLeaf) n = node.left + (p.x[row * p.s.numFeatures + node.feature] < node.value ? 0u : 1u);
        }
        sums[p.s.numClasses > 0 ? tree.classId : 0] += (double)p.globalNodes[n].value;
        if (p.leafIds) p.leafIds[row * p.s.numTrees + tree.origin] = p.globalNodes[n].origin;
      }
      StoreRow(p, row, slice, sums.data());
    }
  }
  return Launched(p.done, stream);
}

hipError_t LaunchBinRows(const float *x, const float *table, uint8_t *ranks, int64_t rows, int numFeatures, int tableDepth,
                         int chunkFeatures, hipStream_t stream) {
  if (rows <= 0) return hipSuccess;
  if (Refused(stream)) return hipErrorLaunchFailure;
  if (chunkFeatures != 64) return hipErrorInvalidValue;
  if (tableDepth < 1 || tableDepth > 255 || ((tableDepth + 1) & tableDepth)) return hipErrorInvalidValue;
  const int64_t rowBlocks = (rows + 63) / 64;
  for (int64_t rb = 0; rb < rowBlocks; ++rb)
    for (int f = 0; f < numFeatures; ++f)
      for (int r = 0; r < 64; ++r) {
        const int64_t row = std::min<int64_t>(rb * 64 + r, rows - 1);
        const float v = x[row * numFeatures + f];
        const float *column = table + ((int64_t)(f / 64) * tableDepth) * 64 + (f % 64);
        int rank = 0;
        for (int step = (tableDepth + 1) / 2; step >= 1; step /= 2)
          if (!(v < column[(int64_t)(rank + step - 1) * 64])) rank += step;
        ranks[(rb * numFeatures + f) * 64 + r] = (uint8_t)rank;
      }
  return hipSuccess;
}

hipError_t LaunchRankRows16(const float *x, const float *tables, const RankFeatureDesc *features, const RankChunkDesc *chunks,
                            int numChunks, uint32_t maxChunkEntries, uint32_t maxChunkFeatures, uint16_t *ranks, int64_t rows,
                            int numFeatures, int rowsPerBlock, hipStream_t stream) {
  if (rows <= 0) return hipSuccess;
  if (Refused(stream)) return hipErrorLaunchFailure;
  if (numChunks < 1 || (size_t)maxChunkEntries * 4 + (size_t)maxChunkFeatures * 1025 * 4 + 16 > 160 * 1024 || rowsPerBlock < 64 ||
      rowsPerBlock % 64 != 0)
    return hipErrorInvalidValue;
  const int64_t RB = rowsPerBlock, pairs = (numFeatures + 2) / 2;
  // the kernel ranks whole row blocks, rounded up to its own tiles of 1024 rows: the buffer has to hold them
  const int64_t rowBlocks = (((rows + RB - 1) / RB * RB + 1023) / 1024 * 1024 + RB - 1) / RB;
  std::vector<char> written((size_t)pairs * 2, 0);
  for (int c = 0; c < numChunks; ++c) {
    const RankChunkDesc ck = chunks[c];
    if (ck.firstFeature % 2 || ck.numFeatures % 2 || ck.firstFeature + ck.numFeatures > (uint32_t)pairs * 2 ||
        ck.tableEntries > maxChunkEntries || ck.numFeatures > maxChunkFeatures)
      std::abort();
    for (uint32_t f = ck.firstFeature; f < ck.firstFeature + ck.numFeatures; ++f) {
      written[f] = 1;
      const RankFeatureDesc fd = features[f];
      const uint32_t entries = (1u << fd.levels) - 1u;
      if (fd.tableOffset + entries > ck.tableEntries) std::abort(); // table outside its chunk
      if ((int)f >= numFeatures && fd.levels != 0) std::abort();     // the pad slots have no table
      const float *table = tables + ck.tableBegin + fd.tableOffset;
      for (int64_t slot = 0; slot < rowBlocks * RB; ++slot) {
        const int64_t row = std::min<int64_t>(slot, rows - 1);
        uint32_t node = 0;
        if (fd.levels) {
          const float v = x[row * numFeatures + f];
          for (uint32_t level = 0; level < fd.levels; ++level) node = 2 * node + (v < table[node] ? 1u : 2u);
        }
        ranks[(((slot / RB) * pairs + f / 2) * RB + slot % RB) * 2 + (f & 1)] = (uint16_t)(node - entries);
      }
    }
  }
  for (char w : written)
    if (!w) std::abort(); // a slot of the tile no chunk fills
  return hipSuccess;
}

namespace {
// A row's class sums -> the outputs asked for (ties go to the larger class id).
void FinishRow(const double *sums, int C, int64_t row, float *out, int8_t *classOut, float *margins, float *probabilities) {
  float best = -INFINITY;
  int bestClass = 0;
  double maxMargin = -INFINITY;
  for (int c = 0; c < C; ++c) {
    const float m = (float)sums[c];
    if (margins) margins[row * C + c] = m;
    if (!(best > m)) best = m, bestClass = c;
    maxMargin = std::max(maxMargin, sums[c]);
  }
  if (classOut) classOut[row] = (int8_t)bestClass;
  if (out) out[row] = (float)bestClass;
  if (probabilities) {
    double z = 0.0;
    for (int c = 0; c < C; ++c) z += std::exp(sums[c] - maxMargin);
    for (int c = 0; c < C; ++c) probabilities[row * C + c] = (float)(std::exp(sums[c] - maxMargin) / z);
  }
}

float FinishMargin(double margin, int transform) { return (float)(transform == 1 ? 1.0 / (1.0 + std::exp(-margin)) : margin); }
} // namespace

hipError_t LaunchFinalize(const FinalizeParams &p, hipStream_t stream) {
  if (p.rows <= 0) return hipSuccess;
  if (Refused(stream)) return hipErrorLaunchFailure;
  const int C = p.numClasses, Cn = std::max(1, C);
  std::vector<double> sums((size_t)Cn);
  for (int64_t row = 0; row < p.rows; ++row) {
    int parts = p.treeSlices;
    if (p.splitBlocks)
      parts = SplitLine{((p.rows + p.rowsPerBlock - 1) / p.rowsPerBlock) * p.groups, p.groups, p.splitBlocks}.Parts(row / p.rowsPerBlock);
    if (parts < 1 || parts > p.treeSlices) std::abort();
    for (int c = 0; c < Cn; ++c) {
      sums[(size_t)c] = p.initialValue;
      for (int s = 0; s < parts; ++s) sums[(size_t)c] += p.partial[((int64_t)s * p.rows + row) * Cn + c];
    }
    if (C == 0) p.out[row] = FinishMargin(sums[0], p.transform);
    else FinishRow(sums.data(), C, row, p.out, p.classOut, p.margins, p.probabilities);
  }
  return Launched(p.done, stream);
}

// The kernel's blocks, lanes and LDS: a row no lane gets to, a leaf outside the block's array, a walk that runs out of the
// blocks (heap memory here) all show.
hipError_t LaunchFewRows(const FewRowsParams &p, hipStream_t stream) {
  if (p.rows <= 0) return hipSuccess;
  if (Refused(stream)) return hipErrorLaunchFailure;
  const FewRowsShape s = ShapeOfFewRows(p.rows, p.numFeatures, p.numTrees, p.numClasses);
  if (p.numTrees < 1 || s.ldsBytes > kFewRowsLds) return hipErrorInvalidValue;
  if (p.numClasses == 0 ? !p.out : !(p.out || p.classOut || p.margins || p.probabilities)) return hipErrorInvalidValue;
  ++shimFewRows;
  const int T = p.numTrees, F = p.numFeatures, R = s.rowsPerBlock, Cn = std::max(1, p.numClasses);
  if (((T * s.leafStride + (size_t)R * F) * 4 + 7) / 8 * 8 + (size_t)R * Cn * 8 > s.ldsBytes) std::abort();
  for (int64_t row0 = 0; row0 < p.rows; row0 += R) {
    const int valid = (int)std::min<int64_t>(R, p.rows - row0);
    std::vector<float> leaves((size_t)T * s.leafStride, std::nanf("")), rowTile(p.x + row0 * F, p.x + (row0 + valid) * F);
    std::vector<double> sums((size_t)R * Cn);
    for (int tid = 0; tid < s.threads; ++tid)
      for (int i = tid; i < valid * T; i += s.threads) {
        const int t = i / valid, r = i - t * valid;
        size_t block = (size_t)t;
        uint32_t slot = 0;
        for (;;) {
          const DeviceFewRowsBlock &b = p.blocks[block];
          if (b.feature[slot] == kFewRowsLeaf) {
            leaves[(size_t)t * s.leafStride + r] = b.value[slot];
            break;
          }
          if (b.feature[slot] >= F) std::abort();
          const uint32_t right = rowTile[(size_t)r * F + b.feature[slot]] < b.value[slot] ? 0u : 1u;
          if (slot < 3) {
            slot = 2 * slot + 1 + right;
            continue;
          }
          const uint32_t exit = 2 * (slot - 3) + right;
          if (!(b.exits >> exit & 1u)) std::abort();
          block = b.firstChild + (uint32_t)__builtin_popcount(b.exits & ((1u << exit) - 1u));
          slot = 0;
        }
      }
    for (int wave = 0; wave < s.threads / 64; ++wave)
      for (int pair = wave; pair < valid * Cn; pair += s.threads / 64) {
        const int r = pair / Cn, c = pair - r * Cn;
        double margin = p.initialValue;
        for (int t = p.numClasses > 0 ? p.classBegin[c] : 0, end = p.numClasses > 0 ? p.classBegin[c + 1] : T; t < end; ++t)
          margin += (double)leaves[(size_t)t * s.leafStride + r];
        if (p.numClasses == 0) p.out[row0 + r] = FinishMargin(margin, p.transform);
        else sums[(size_t)pair] = margin;
      }
    for (int tid = 0; p.numClasses > 0 && tid < s.threads; ++tid)
      for (int r = tid; r < valid; r += s.threads)
        FinishRow(sums.data() + (size_t)r * Cn, Cn, row0 + r, p.out, p.classOut, p.margins, p.probabilities);
  }
  return Launched(p.done, stream);
}

hipError_t LaunchRankStream(const RankStreamParams &p, hipStream_t stream) {
  if (p.rows <= 0) return hipSuccess;
  if (Refused(stream)) return hipErrorLaunchFailure;
  const int waves = StreamWaves(p.numFeatures), F = p.numFeatures;
  if (waves < 1 || F > kStreamMaxFeatures || p.numBundles < 1 || (p.chains != 2 && p.chains != 4) || p.slices < 1 || p.slices > 65535)
    return hipErrorInvalidValue;
  if (p.slices > 1 ? !p.partial : !p.out) return hipErrorInvalidValue;
  if ((((size_t)(F + 1) * kStreamRows + 15) & ~(size_t)15) + (size_t)waves * 2 * kStreamBundleBytes > 160 * 1024) return hipErrorInvalidValue;
  ++shimStreams;
  for (int slice = 0; slice < p.slices; ++slice) {
    const int first = (int)((int64_t)p.numBundles * slice / p.slices), last = (int)((int64_t)p.numBundles * (slice + 1) / p.slices);
    for (int64_t row = 0; row < p.rows; ++row) {
      double sum = 0.0;
      for (int b = first; b < last; ++b) {
        const uint32_t begin = p.bundles[b];
        if (begin % 4) std::abort();
        DeviceStreamHead heads[2];
        std::memcpy(heads, p.words + begin, sizeof(heads));
        const uint32_t depth = heads[0].depth, words = heads[0].words;
        if (depth < 1 || heads[1].depth != depth || heads[1].words != words || words * 4 > kStreamBundleBytes) std::abort();
        if (b + 1 < p.numBundles && p.bundles[b + 1] != begin + words) std::abort();
        if (p.words[begin + kStreamBundleBytes / 4 - 1] == 0xFFFFFFFFu) std::abort(); // (the copy reads that far)
        for (int k = 0; k < 2 * p.chains; ++k) {
          const uint32_t root = heads[k & 1].roots[k / 2] / 4u;
          if (root % 2) std::abort(); // (children are read two words at a time)
          uint32_t at = 0;
          for (uint32_t d = 0; d < depth; ++d) {
            // a node outside the bundle's trees (the root is the head's; a leaf that is a tree has it as a word too)
            if (d > 0 && (root + at < kStreamHeadWords || root + at >= words)) std::abort();
            const uint32_t node = d > 0 ? p.words[begin + root + at] : heads[k & 1].rootWords[k / 2], f = node >> 5 & 0x7FFu;
            if (d > 0 && at == 0 && node != heads[k & 1].rootWords[k / 2]) std::abort();
            if ((int)f > F || (node & 31u)) std::abort();
            const uint32_t rank = (int)f == F ? 0u : p.ranks[((row / 64) * F + f) * 64 + row % 64];
            at = 2 * (node >> 16 & 0xFFu) + (rank < node >> 24 ? 0u : 1u);
          }
          sum += (double)p.values[heads[k & 1].valueBegin[k / 2] + at];
        }
      }
      if (p.slices > 1) p.partial[(int64_t)slice * p.rows + row] = sum;
      else p.out[row] = FinishMargin(p.initialValue + sum, p.transform);
    }
  }
  return Launched(p.done, stream);
}

} // namespace tbamd
