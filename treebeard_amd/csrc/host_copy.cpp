#include "host_copy.h"

#include <algorithm>
#include <cstring>
#include <emmintrin.h>

namespace tbamd {

namespace {
constexpr size_t kPieceBytes = (size_t)128 << 10;  // what a thread takes at a time: some 10 us
constexpr size_t kLoneBytes = (size_t)1 << 20;     // below, waking the pool takes longer than it saves

// memcpy with stores that leave the caches alone (they are ordered by the fence)
void StreamedCopy(char *dst, const char *src, size_t bytes) {
  const size_t head = std::min(bytes, (size_t)(-reinterpret_cast<uintptr_t>(dst) & 63));
  std::memcpy(dst, src, head);
  dst += head, src += head, bytes -= head;
  for (; bytes >= 64; dst += 64, src += 64, bytes -= 64) {
    __m128i line[4];
    for (int i = 0; i < 4; ++i) line[i] = _mm_loadu_si128(reinterpret_cast<const __m128i *>(src) + i);
    for (int i = 0; i < 4; ++i) _mm_stream_si128(reinterpret_cast<__m128i *>(dst) + i, line[i]);
  }
  std::memcpy(dst, src, bytes);
  _mm_sfence();
}
} // namespace

ParallelCopier::ParallelCopier(int threads) {
  for (int i = 1; i < std::max(1, threads); ++i) m_workers.emplace_back([this] { Worker(); });
}

ParallelCopier::~ParallelCopier() {
  Finish();
  {
    std::lock_guard<std::mutex> lock(m_mutex);
    m_stop = true;
  }
  m_wake.notify_all();
  for (auto &t : m_workers) t.join();
}

// Copies the next piece of the parts up to `lastPart`, if one is left.  Called and returns with the lock held.
bool ParallelCopier::CopySome(std::unique_lock<std::mutex> &lock, size_t lastPart) {
  if (m_next >= m_parts.size() || m_next > lastPart) return false;
  Part &part = m_parts[m_next];
  const size_t begin = m_offset, bytes = std::min(kPieceBytes, part.bytes - begin);
  m_offset += bytes;
  if (m_offset == part.bytes) ++m_next, m_offset = 0;
  m_copying.fetch_add(1, std::memory_order_relaxed);
  lock.unlock();
  if (part.streamed) StreamedCopy(part.dst + begin, part.src + begin, bytes);
  else std::memcpy(part.dst + begin, part.src + begin, bytes);
  part.left.fetch_sub(bytes, std::memory_order_release);
  m_copying.fetch_sub(1, std::memory_order_release);
  lock.lock();
  return true;
}

void ParallelCopier::Worker() {
  std::unique_lock<std::mutex> lock(m_mutex);
  while (!m_stop) {
    if (m_next < m_parts.size() && m_sleeping > 0) m_wake.notify_one(); // (one wakes the next: no thread wakes all)
    if (CopySome(lock, SIZE_MAX)) continue;
    ++m_sleeping;
    m_wake.wait(lock);
    --m_sleeping;
  }
}

void ParallelCopier::Append(void *dst, const void *src, size_t bytes, bool streamed) {
  bool wake;
  {
    std::lock_guard<std::mutex> lock(m_mutex);
    m_parts.emplace_back(static_cast<char *>(dst), static_cast<const char *>(src), bytes, streamed);
    if (bytes == 0) return;
    wake = m_sleeping > 0;
  }
  if (wake) m_wake.notify_one();
}

void ParallelCopier::Await(size_t index) {
  Part *part;
  {
    std::unique_lock<std::mutex> lock(m_mutex);
    while (CopySome(lock, index)) {}
    part = &m_parts[index];
  }
  while (part->left.load(std::memory_order_acquire) != 0) std::this_thread::yield(); // (a piece of some 10 us)
}

void ParallelCopier::Finish() {
  {
    std::lock_guard<std::mutex> lock(m_mutex);
    m_next = m_parts.size();
    m_offset = 0;
  }
  while (m_copying.load(std::memory_order_acquire) != 0) std::this_thread::yield();
  std::lock_guard<std::mutex> lock(m_mutex);
  m_parts.clear();
  m_next = 0;
}

void ParallelCopier::Copy(void *dst, const void *src, size_t bytes) {
  if (m_workers.empty() || bytes < kLoneBytes) {
    if (bytes) std::memcpy(dst, src, bytes);
    return;
  }
  Append(dst, src, bytes, false);
  Await(0);
  Finish();
}

} // namespace tbamd
