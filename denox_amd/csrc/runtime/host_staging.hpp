// Transfers between pageable host memory and the device for the blocking entry point.
//
// The driver moves a pageable array in one thread through a staging buffer of its own: 37 MB up take 1.40 ms where the link
// needs 0.66, 12 MB down 0.75 ms for 0.23.  Here several threads copy between the caller's array and page-locked memory, chunk by
// chunk, while the chunks before (up) or behind (down) are on the link.
// U-Net at 1920 x 1080 from and to pageable arrays, one blocking call: 2.70 - 2.90 ms, 1.94 - 1.97 so.
#pragma once
#include <hip/hip_runtime_api.h>
#include <cstddef>
#include <cstdint>
#include <vector>

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
  // Before the first transfer of a call: the bytes that will be staged in all, so that a download need not wait for room.
  void prepare(uint64_t bytes, hipStream_t s) { reserve(bytes, s); }
  // Enqueues the copy on `s`; returns when the whole array has been read.
  void upload(void *device, const void *host, uint64_t bytes, hipStream_t s);
  // Waits for what is enqueued on `s` and copies; returns when the whole array has been written.
  void download(void *host, const void *device, uint64_t bytes, hipStream_t s);

private:
  void reserve(uint64_t bytes, hipStream_t s);
  uint8_t *m_pinned = nullptr; // at most kMaxBytes, kept for the life of its owner
  uint64_t m_capacity = 0, m_used = 0; // [0, m_used): chunks that the link may still be reading
  std::vector<hipEvent_t> m_events;
};

} // namespace denox::runtime
