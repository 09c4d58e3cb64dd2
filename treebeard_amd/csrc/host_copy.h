// Copies between pageable host memory and pinned staging buffers with several threads: one core moves
// about 10 GB/s out of memory, less than the link to the device, so the host-buffer entry point hands
// the rows of a call to a small pool that lives as long as the runner.
#pragma once
#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstddef>
#include <cstdint>
#include <deque>
#include <mutex>
#include <thread>
#include <vector>

namespace tbamd {

// How a host batch is cut: pieces of about 4 MB (73 us of the link, which cover the 10 us the calling thread needs for a piece),
// at least 1024 rows (fewer take the kernels as long) and `leastRows` (what the kernels need to work at their rate; two thirds of
// the batch at most, so that something overlaps), as long as those fit 16 MB; a quarter and half a piece first, because
// nothing overlaps their copies, and what is left at the end as two thirds and one third, because nothing overlaps the last
// piece's kernels.  The pieces take turns in `slots` pinned buffers: eight of 4 MB, fewer of larger ones (four are what two
// copies under way, a piece in its kernels and one being filled need), so that they pin 32 MB, 64 for the widest rows.
constexpr size_t kHostPieceBytes = (size_t)4 << 20, kHostPartBytes = (size_t)1 << 20;
constexpr int kHostSlots = 8;
struct HostPieces {
  int64_t rows, most, count; // `most`: rows of the largest piece
  int64_t slots;
  HostPieces(int64_t allRows, size_t rowBytes, int64_t leastRows = 0) : rows(allRows) {
    const int64_t fit = (int64_t)((4 * kHostPieceBytes) / rowBytes);
    most = std::min(std::max<int64_t>({(int64_t)(kHostPieceBytes / rowBytes), 1024, std::min(leastRows, rows * 2 / 3)}), fit);
    most = most >= 256 ? most / 256 * 256 : std::max<int64_t>(4, most); // (rows of 4 MB and more: four of them)
    slots = std::max<int64_t>(4, std::min<int64_t>(kHostSlots, (int64_t)(kHostSlots * kHostPieceBytes / ((size_t)most * rowBytes))));
    if (rows <= most) most = rows, count = 1;
    else count = 2 + (rows - most / 4 * 3 + most - 1) / most;
  }
  int64_t End(int64_t p) const {
    if (p >= count - 1) return rows;
    if (p == 0) return most / 4;
    const int64_t begin = most / 4 * 3 + (p - 2) * most;
    return p == count - 2 && p > 1 ? begin + std::min(most, ((rows - begin) * 2 / 3 + 63) / 64 * 64) : begin + most;
  }
  int64_t Begin(int64_t p) const { return p == 0 ? 0 : End(p - 1); }
  int64_t Rows(int64_t p) const { return End(p) - Begin(p); }
};

class ParallelCopier {
public:
  explicit ParallelCopier(int threads); // the calling thread counts as one of them
  ~ParallelCopier();
  ParallelCopier(const ParallelCopier &) = delete;
  ParallelCopier &operator=(const ParallelCopier &) = delete;
  // memcpy(dst, src, bytes), shared by the pool; returns when it is done.
  void Copy(void *dst, const void *src, size_t bytes);
  // A copy in parts, which the pool does in order and ahead of the caller: Append() hands over the next part (its
  // destination is free; `streamed`: written past the caches), Await() returns once part i is written, working on the
  // parts up to it meanwhile, and Finish() ends the copy; parts that nobody awaited may then be left undone.  One copy
  // at a time.
  void Append(void *dst, const void *src, size_t bytes, bool streamed);
  void Await(size_t part);
  void Finish();
  int Threads() const { return (int)m_workers.size() + 1; }

private:
  struct Part {
    Part(char *to, const char *from, size_t size, bool past) : dst(to), src(from), bytes(size), left(size), streamed(past) {}
    char *dst;
    const char *src;
    size_t bytes;
    std::atomic<size_t> left; // bytes not yet written
    bool streamed;
  };
  void Worker();
  bool CopySome(std::unique_lock<std::mutex> &lock, size_t lastPart);
  std::vector<std::thread> m_workers;
  std::mutex m_mutex;
  std::condition_variable m_wake;
  std::deque<Part> m_parts; // (a deque: parts stay where they are while others are appended)
  size_t m_next = 0, m_offset = 0; // the next piece to copy
  int m_sleeping = 0;
  std::atomic<int> m_copying{0};
  bool m_stop = false;
};

} // namespace tbamd
