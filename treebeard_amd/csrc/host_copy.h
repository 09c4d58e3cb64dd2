// Copies between pageable host memory and pinned staging buffers with several threads: one core moves
// about 10 GB/s out of memory, less than the link to the device, so the host-buffer entry point hands
// the rows of a call to a small pool that lives as long as the runner.
#pragma once
#include <atomic>
#include <condition_variable>
#include <cstddef>
#include <cstdint>
#include <deque>
#include <mutex>
#include <thread>
#include <vector>

namespace tbamd {

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
