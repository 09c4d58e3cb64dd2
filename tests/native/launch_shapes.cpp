// The host-side arithmetic that the launchers and the runner share (kernels.h, host_copy.h), over its whole range.
#include "host_copy.h"
#include "kernels.h"

#include <cstdio>
#include <vector>

using namespace tbamd;

static int gFailures = 0;
#define EXPECT(cond, ...)                                                                                              \
  do {                                                                                                                 \
    if (!(cond) && ++gFailures < 20) std::printf("FAILED %s: ", #cond), std::printf(__VA_ARGS__), std::printf("\n"); \
  } while (0)

// Every forest: the batches up to its limit fit a block's LDS and its lanes (a lane per row finishes the classes), and no
// wave adds more sums than 0.4 us each are worth.
static void FewRows() {
  for (int classes : {0, 2, 3, 6, 12, 40, 128})
    for (int trees = 1; trees <= 1200; trees += trees < 40 ? 1 : 97)
      for (int features : {1, 4, 28, 600, 2047, 20000})
        for (int depth : {0, 1, 3, 6, 8, 14, 30}) {
          const int64_t limit = FewRowsLimit(features, trees, classes, depth);
          EXPECT(limit >= 0 && limit <= kFewRowsWork, "%d classes %d trees %d features depth %d", classes, trees, features, depth);
          for (int64_t rows : {(int64_t)1, limit / 3, limit - 1, limit}) {
            if (rows < 1 || rows > limit) continue;
            const FewRowsShape s = ShapeOfFewRows(rows, features, trees, classes);
            const int64_t sums = (int64_t)s.rowsPerBlock * (classes ? classes : 1);
            EXPECT(s.threads % 64 == 0 && s.threads <= 1024 && s.ldsBytes <= kFewRowsLds, "%d classes %d trees %d features depth %d: %lld rows",
                   classes, trees, features, depth, (long long)rows);
            EXPECT(s.rowsPerBlock <= s.threads, "%d classes %d trees %d features depth %d: %lld rows, %d a block of %d lanes", classes, trees, features,
                   depth, (long long)rows, s.rowsPerBlock, s.threads);
            EXPECT(rows < limit || (sums - 1) / (s.threads / 64) * 0.4 <= 6.5 + 1.1 * classes, "%d classes %d trees %d features depth %d: %lld rows", classes,
                   trees, features, depth, (long long)rows);
          }
        }
}

// Parts of the line of row blocks x groups against the owners counted one by one.
static void SplitLines() {
  for (int64_t rowBlocks = 1; rowBlocks <= 70; rowBlocks += rowBlocks < 9 ? 1 : 7)
    for (int groups = 1; groups <= 40; groups += groups < 6 ? 1 : 5)
      for (int64_t blocks = 1; blocks <= rowBlocks * groups; blocks += blocks < 12 ? 1 : 1 + rowBlocks * groups / 23) {
        const SplitLine line{rowBlocks * groups, groups, (int)blocks};
        EXPECT(line.FirstUnit(0) == 0 && line.FirstUnit(blocks) == line.units, "%d groups %lld blocks", groups, (long long)blocks);
        std::vector<int64_t> owner((size_t)line.units, -1);
        for (int64_t b = 0; b < blocks; ++b)
          for (int64_t u = line.FirstUnit(b); u < line.FirstUnit(b + 1); ++u) owner[(size_t)u] = b;
        for (int64_t r = 0; r < rowBlocks; ++r) {
          const int64_t first = owner[(size_t)(r * groups)], last = owner[(size_t)((r + 1) * groups - 1)];
          EXPECT(first == line.FirstBlock(r) && last - first + 1 == line.Parts(r) && line.Parts(r) <= SplitLine::Slots(blocks, rowBlocks),
                 "row block %lld of %lld, %d groups, %lld blocks", (long long)r, (long long)rowBlocks, groups, (long long)blocks);
        }
      }
}

// Every width of the form: the ranks and two bundles a wave fit LDS, and the slices never outnumber the bundles.
static void Streams() {
  for (int features = 1; features <= kStreamMaxFeatures; ++features) {
    const int waves = StreamWaves(features);
    EXPECT(waves >= 1 && waves <= kStreamMaxWaves && ((features + 1) * kStreamRows + 15) / 16 * 16 + waves * 2 * (int)kStreamBundleBytes <= 160 * 1024,
           "%d features: %d waves", features, waves);
    for (int bundles : {1, 2, 31, 125, 4000})
      for (int64_t rows : {(int64_t)1, (int64_t)33, (int64_t)5000, (int64_t)1 << 20}) {
        const int slices = RankStreamSlices(rows, features, bundles, 256);
        EXPECT(slices >= 1 && slices <= 64 && (slices == 1 || slices * 2 * waves <= bundles), "%d features, %d bundles: %d slices", features, bundles, slices);
      }
  }
}

// Host batches: pieces follow each other without gaps, none is empty or larger than its buffer, a buffer's piece has been
// drained before the next one is copied into it, and the buffers of a runner stay under 64 MB (four rows at least each).
static void HostBatches() {
  for (size_t features : {1, 3, 8, 28, 250, 1000, 1024, 1025, 2000, 3000, 4096, 5003, 16000, 16384, 16385, 20000, 65535, 300000, 1 << 20, 3000000})
    for (int64_t scale = 1; scale <= 4096; scale += scale < 24 ? 1 : scale / 3)
      for (int64_t extra : {-1, 0, 1, 63, 64, 255}) {
        const size_t rowBytes = features * 4;
        const int64_t least = scale % 3 == 0 ? 0 : 6144 << scale % 7; // (what a launch plan asks for)
        const int64_t step = HostPieces((int64_t)1 << 40, rowBytes, least).most, rows = scale * step / 8 + extra;
        if (rows < 1) continue;
        const HostPieces p(rows, rowBytes, least);
        EXPECT(step >= std::min<int64_t>(least / 256 * 256, ((int64_t)16 << 20) / (int64_t)rowBytes / 256 * 256), "%zu features: pieces of %lld rows for %lld",
               features, (long long)step, (long long)least);
        EXPECT(p.count >= 1 && p.slots >= 4 && p.slots <= kHostSlots && p.slots / 2 - 1 + 2 <= p.slots - 1, "%zu features %lld rows", features, (long long)rows);
        EXPECT((size_t)(p.slots * p.most) * rowBytes <= (size_t)64 << 20 || p.most <= 4, "%zu features %lld rows: %lld buffers of %lld rows", features,
               (long long)rows, (long long)p.slots, (long long)p.most);
        int64_t end = 0;
        for (int64_t i = 0; i < p.count; ++i) {
          EXPECT(p.Begin(i) == end && p.Rows(i) >= 1 && p.Rows(i) <= p.most, "%zu features %lld rows, piece %lld: %lld rows", features, (long long)rows,
                 (long long)i, (long long)p.Rows(i));
          end = p.End(i);
        }
        EXPECT(end == rows, "%zu features %lld rows", features, (long long)rows);
      }
}

int main() {
  HostBatches();
  FewRows();
  SplitLines();
  Streams();
  if (gFailures) return 1;
  std::printf("ok\n");
  return 0;
}
