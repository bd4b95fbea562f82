// Transfers between pageable host memory and the device for the blocking entry point.
//
// The driver moves a pageable array in one thread through a staging buffer of its own: 37 MB up take 1.40 ms where the link
// needs 0.66, 12 MB down 0.75 ms for 0.23.  Here several threads copy between the caller's array and a ring of page-locked chunks
// while the chunks before (up) or behind (down) are on the link; an event behind each says when its slot can be used again.
// Chunk and ring: a transfer and its event cost ~15 us beside the link's 75 for 4 MiB (2 MiB chunks: 0.15 ms more per call), and
// page-locked memory costs 0.1 ms per MiB when it is first touched, which the first call pays.
// U-Net at 1920 x 1080 (0.59 ms of kernels) from and to pageable arrays, one blocking call: 2.85 ms through the driver, 2.04 so; a
// process's first 12.5 and 3.9, a further context's first 7.5 and 3.3.  (A buffer of 64 MiB: 1.98, first 5.6.)
#pragma once
#include <hip/hip_runtime_api.h>
#include <cstddef>
#include <cstdint>

namespace denox::runtime {

class HostStaging {
public:
  HostStaging() = default;
  ~HostStaging();
  HostStaging(const HostStaging &) = delete;
  HostStaging &operator=(const HostStaging &) = delete;

  // Whether a transfer of `bytes` at `host` gains from staging: large enough to pay for the threads, and not page-locked
  // already (then the link can read it directly).
  static bool worthwhile(const void *host, uint64_t bytes);
  // Page-locked memory is there (made on the first call).  false: it cannot be had, transfer directly.
  bool ready();
  // Enqueues the copy on `s`; returns when the whole array has been read.
  void upload(void *device, const void *host, uint64_t bytes, hipStream_t s);
  // Waits for what is enqueued on `s` and copies; returns when the whole array has been written.
  void download(void *host, const void *device, uint64_t bytes, hipStream_t s);

  static constexpr uint64_t kChunk = 4ull << 20; // one link transfer
  static constexpr size_t kSlots = 4;            // of the ring

private:
  void begin(hipStream_t s);
  bool idle(size_t slot, bool wait);
  void release();
  uint8_t *m_pinned = nullptr;      // kSlots chunks, used in turn, kept for the life of their owner
  hipEvent_t m_events[kSlots] = {}; // behind the last transfer of a slot
  bool m_busy[kSlots] = {};         // that event has not been waited for
  uint64_t m_next = 0;              // slot of the next transfer's first chunk
  bool m_unsettled = false;         // a transfer has begun and not ended
};

} // namespace denox::runtime
