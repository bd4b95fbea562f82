#include "host_staging.hpp"
#include "runtime.hpp"
#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstring>
#include <functional>
#include <mutex>
#include <thread>

namespace denox::runtime {

namespace {

constexpr uint64_t kWorthwhile = 4ull << 20; // below, starting the threads costs what they save
constexpr unsigned kThreads = 8;             // 37 MB: 1.35 ms with one thread, 0.50 with four, 0.38 with eight, no less with twelve

constexpr uint64_t kChunk = HostStaging::kChunk;
constexpr uint64_t kPiece = 128ull << 10; // what a thread copies at a time: all of them share a chunk, so that the first one is soon on the link

// Threads that copy an array piece by piece, in order; `copy(offset, bytes)` runs for each piece exactly once.
// gate: the chunks [0, gate) may be copied (none at first).
class Copiers {
public:
  Copiers(uint64_t bytes, std::function<void(uint64_t, uint64_t)> copy) : m_bytes(bytes), m_copy(std::move(copy)) {
    for (uint64_t at = 0; at < bytes; at += kChunk) m_left.push_back(pieces(std::min(kChunk, bytes - at)));
    const unsigned hw = std::max(1u, std::thread::hardware_concurrency());
    const uint64_t n = std::min<uint64_t>(pieces(bytes), std::min(kThreads, hw));
    m_threads.reserve(n);
    for (uint64_t t = 0; t < n; ++t) {
      try { // (the vector's memory is there; the thread and its state may be refused)
        m_threads.emplace_back([this] {
          for (;;) {
            const uint64_t at = m_next.fetch_add(kPiece);
            if (at >= m_bytes) return;
            {
              std::unique_lock<std::mutex> l(m_mutex);
              m_cv.wait(l, [&] { return m_stop || at / kChunk < m_gate; });
              if (m_stop) return;
            }
            m_copy(at, std::min(kPiece, m_bytes - at));
            std::lock_guard<std::mutex> l(m_mutex);
            if (--m_left[at / kChunk] == 0) m_cv.notify_all();
          }
        });
      } catch (...) {
        break; // those that started do all the work; without any, wait() does it
      }
    }
  }
  ~Copiers() {
    {
      std::lock_guard<std::mutex> l(m_mutex);
      m_stop = true;
      m_cv.notify_all();
    }
    for (auto &t : m_threads) t.join();
  }
  void open(uint64_t gate) {
    std::lock_guard<std::mutex> l(m_mutex);
    m_gate = gate;
    m_cv.notify_all();
  }
  // chunk i, which is behind the gate, has been copied
  void wait(uint64_t i) {
    if (m_threads.empty()) {
      if (m_left[i]) m_copy(i * kChunk, std::min(kChunk, m_bytes - i * kChunk));
      m_left[i] = 0;
      return;
    }
    std::unique_lock<std::mutex> l(m_mutex);
    m_cv.wait(l, [&] { return m_left[i] == 0; });
  }
  bool done(uint64_t i) {
    std::lock_guard<std::mutex> l(m_mutex);
    return m_left[i] == 0;
  }

private:
  static uint64_t pieces(uint64_t bytes) { return (bytes + kPiece - 1) / kPiece; }
  const uint64_t m_bytes;
  std::function<void(uint64_t, uint64_t)> m_copy;
  std::mutex m_mutex;
  std::condition_variable m_cv;
  std::vector<uint64_t> m_left; // pieces of a chunk that have not been copied
  uint64_t m_gate = 0;
  bool m_stop = false;
  std::atomic<uint64_t> m_next{0};
  std::vector<std::thread> m_threads;
};

} // namespace

HostStaging::~HostStaging() { release(); }

void HostStaging::release() {
  for (hipEvent_t &e : m_events) {
    if (e) (void)hipEventDestroy(e);
    e = nullptr;
  }
  if (m_pinned) (void)hipHostFree(m_pinned);
  m_pinned = nullptr;
}

bool HostStaging::worthwhile(const void *host, uint64_t bytes) {
  if (bytes < kWorthwhile) return false;
  hipPointerAttribute_t a;
  const hipError_t e = hipPointerGetAttributes(&a, host);
  if (e != hipSuccess) {
    (void)hipGetLastError(); // memory the runtime does not know: pageable
    return true;
  }
  return a.type == hipMemoryTypeUnregistered;
}

bool HostStaging::ready() {
  if (m_pinned) return true;
  void *p = nullptr;
  bool ok = hipHostMalloc(&p, kSlots * kChunk, hipHostMallocDefault) == hipSuccess;
  if (ok) m_pinned = static_cast<uint8_t *>(p);
  for (size_t i = 0; ok && i < kSlots; ++i) ok = hipEventCreateWithFlags(&m_events[i], hipEventDisableTiming) == hipSuccess;
  if (ok) return true;
  (void)hipGetLastError();
  release();
  return false;
}

void HostStaging::begin(hipStream_t s) {
  if (m_unsettled) { // a transfer ended half-way: the link may still read or write any slot
    hipCheck(hipStreamSynchronize(s), "hipStreamSynchronize");
    std::fill(std::begin(m_busy), std::end(m_busy), false);
  }
  m_unsettled = true;
}

// Slot `i` can be written again: its last transfer has passed, or `wait` for that.
bool HostStaging::idle(size_t i, bool wait) {
  if (!m_busy[i]) return true;
  if (wait) hipCheck(hipEventSynchronize(m_events[i]), "hipEventSynchronize");
  else {
    const hipError_t e = hipEventQuery(m_events[i]);
    if (e == hipErrorNotReady) return false;
    hipCheck(e, "hipEventQuery");
  }
  m_busy[i] = false;
  return true;
}

void HostStaging::upload(void *device, const void *host, uint64_t bytes, hipStream_t s) {
  begin(s);
  const uint8_t *src = static_cast<const uint8_t *>(host);
  uint8_t *dst = static_cast<uint8_t *>(device);
  const uint64_t chunks = (bytes + kChunk - 1) / kChunk, first = m_next;
  auto size = [=](uint64_t i) { return std::min(kChunk, bytes - i * kChunk); };
  auto slot = [=](uint64_t i) { return static_cast<size_t>((first + i) % kSlots); };
  uint8_t *ring = m_pinned;
  uint64_t open = 0; // chunks whose slot may be written
  {
    Copiers copiers(bytes, [=](uint64_t at, uint64_t n) { std::memcpy(ring + slot(at / kChunk) * kChunk + at % kChunk, src + at, n); });
    for (uint64_t i = 0; i < chunks; ++i) {
      while (open < chunks && open < i + kSlots && idle(slot(open), open == i)) ++open;
      copiers.open(open);
      copiers.wait(i);
      hipCheck(hipMemcpyAsync(dst + i * kChunk, ring + slot(i) * kChunk, size(i), hipMemcpyHostToDevice, s), "hipMemcpyAsync(input)");
      hipCheck(hipEventRecord(m_events[slot(i)], s), "hipEventRecord");
      m_busy[slot(i)] = true;
    }
  }
  m_next = (first + chunks) % kSlots;
  m_unsettled = false;
}

void HostStaging::download(void *host, const void *device, uint64_t bytes, hipStream_t s) {
  begin(s);
  uint8_t *dst = static_cast<uint8_t *>(host);
  const uint8_t *src = static_cast<const uint8_t *>(device);
  const uint64_t chunks = (bytes + kChunk - 1) / kChunk, first = m_next;
  auto size = [=](uint64_t i) { return std::min(kChunk, bytes - i * kChunk); };
  auto slot = [=](uint64_t i) { return static_cast<size_t>((first + i) % kSlots); };
  const uint8_t *ring = m_pinned;
  uint64_t sent = 0;
  auto send = [&] { // (an upload that still reads the slot comes first in stream order)
    hipCheck(hipMemcpyAsync(m_pinned + slot(sent) * kChunk, src + sent * kChunk, size(sent), hipMemcpyDeviceToHost, s), "hipMemcpyAsync(output)");
    hipCheck(hipEventRecord(m_events[slot(sent)], s), "hipEventRecord");
    m_busy[slot(sent)] = true;
    ++sent;
  };
  while (sent < std::min<uint64_t>(chunks, kSlots)) send();
  {
    // the threads start while the kernels still run
    Copiers copiers(bytes, [=](uint64_t at, uint64_t n) { std::memcpy(dst + at, ring + slot(at / kChunk) * kChunk + at % kChunk, n); });
    for (uint64_t i = 0; i < chunks; ++i) {
      if (sent == i) copiers.wait(i - kSlots); // every slot is waiting to be copied out
      while (sent < chunks && sent < i + kSlots && copiers.done(sent - kSlots)) send();
      (void)idle(slot(i), true);
      copiers.open(i + 1);
    }
    for (uint64_t i = 0; i < chunks; ++i) copiers.wait(i);
  }
  m_next = (first + chunks) % kSlots;
  m_unsettled = false;
}

} // namespace denox::runtime
