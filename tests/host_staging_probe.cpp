// Test program for denox_amd/csrc/runtime/host_staging.cpp without a GPU: the HIP calls it makes are stood in for by one
// "stream" thread that runs copies and events in order, as late as it is told to, and by allocations that fail on demand.
// usage: host_staging_probe CASE; prints "ok" or what went wrong.
#include "../denox_amd/csrc/runtime/host_staging.cpp"
#include <atomic>
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <deque>
#include <new>
#include <random>

namespace {
std::mutex g_mutex;
std::condition_variable g_cv;
struct Work { std::function<void()> run; };
std::deque<Work> g_queue;
uint64_t g_enqueued = 0, g_finished = 0;
std::atomic<int> g_delayUs{0}, g_failPinned{0}, g_failEvents{0}, g_failCopy{-1}, g_pinned{0}, g_events{0};
std::atomic<long> g_failNew{-1}; // operator new fails from the n-th call on
struct Event { uint64_t at = 0; };

void stream() {
  for (;;) {
    Work w;
    {
      std::unique_lock<std::mutex> l(g_mutex);
      g_cv.wait(l, [] { return !g_queue.empty(); });
      w = std::move(g_queue.front());
      g_queue.pop_front();
    }
    if (!w.run) return;
    if (const int d = g_delayUs) std::this_thread::sleep_for(std::chrono::microseconds(d));
    w.run();
    std::lock_guard<std::mutex> l(g_mutex);
    ++g_finished;
    g_cv.notify_all();
  }
}
void push(std::function<void()> f) {
  std::lock_guard<std::mutex> l(g_mutex);
  const bool work = static_cast<bool>(f);
  g_queue.push_back(Work{std::move(f)});
  if (work) ++g_enqueued;
  g_cv.notify_all();
}
} // namespace

void *operator new(size_t n) {
  if (g_failNew >= 0 && g_failNew-- == 0) {
    g_failNew = 0; // and every one after it
    throw std::bad_alloc();
  }
  if (void *p = std::malloc(n ? n : 1)) return p;
  throw std::bad_alloc();
}
void operator delete(void *p) noexcept { std::free(p); }
void operator delete(void *p, size_t) noexcept { std::free(p); }

extern "C" {
hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
  if (g_failPinned) return hipErrorOutOfMemory;
  *p = std::malloc(n);
  ++g_pinned;
  return hipSuccess;
}
hipError_t hipHostFree(void *p) {
  std::free(p);
  --g_pinned;
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) {
  if (g_failEvents && g_events >= 2) return hipErrorOutOfMemory;
  *e = reinterpret_cast<hipEvent_t>(new Event);
  ++g_events;
  return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e) {
  delete reinterpret_cast<Event *>(e);
  --g_events;
  return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t) {
  std::lock_guard<std::mutex> l(g_mutex);
  reinterpret_cast<Event *>(e)->at = g_enqueued;
  return hipSuccess;
}
hipError_t hipEventQuery(hipEvent_t e) {
  std::lock_guard<std::mutex> l(g_mutex);
  return g_finished >= reinterpret_cast<Event *>(e)->at ? hipSuccess : hipErrorNotReady;
}
hipError_t hipEventSynchronize(hipEvent_t e) {
  std::unique_lock<std::mutex> l(g_mutex);
  const uint64_t at = reinterpret_cast<Event *>(e)->at;
  g_cv.wait(l, [&] { return g_finished >= at; });
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) {
  std::unique_lock<std::mutex> l(g_mutex);
  g_cv.wait(l, [] { return g_finished == g_enqueued; });
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t) {
  if (g_failCopy >= 0 && g_failCopy-- == 0) return hipErrorUnknown;
  push([=] { std::memcpy(d, s, n); });
  return hipSuccess;
}
hipError_t hipPointerGetAttributes(hipPointerAttribute_t *, const void *) { return hipErrorInvalidValue; }
hipError_t hipGetLastError() { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "error"; }
}

namespace denox::runtime {
void hipCheck(hipError_t e, const char *what) {
  if (e != hipSuccess) fail(Status::HipError, what);
}
} // namespace denox::runtime

using denox::runtime::HostStaging;
static std::mt19937 rng(1);
static std::vector<uint8_t> bytes(uint64_t n) {
  std::vector<uint8_t> v(n);
  for (auto &b : v) b = static_cast<uint8_t>(rng());
  return v;
}
static void need(bool ok, const char *what) {
  if (ok) return;
  std::printf("wrong: %s\n", what);
  std::fflush(stdout);
  std::_Exit(1);
}

// uploads of the given sizes behind one another, then the same arrays down again
static void roundTrip(HostStaging &st, const std::vector<uint64_t> &sizes) {
  need(st.ready(), "ready");
  std::vector<std::vector<uint8_t>> host, device;
  for (uint64_t n : sizes) {
    host.push_back(bytes(n));
    device.emplace_back(n);
    std::vector<uint8_t> mine = host.back();
    st.upload(device.back().data(), mine.data(), n, nullptr);
    std::fill(mine.begin(), mine.end(), uint8_t(0)); // the caller may reuse its array at once
  }
  for (size_t i = 0; i < sizes.size(); ++i) {
    std::vector<uint8_t> back(sizes[i]);
    st.download(back.data(), device[i].data(), sizes[i], nullptr);
    need(back == host[i], "array came back changed");
  }
}

int main(int argc, char **argv) {
  const std::string c = argc > 1 ? argv[1] : "";
  std::thread worker(stream);
  const uint64_t M = 1ull << 20, C = HostStaging::kChunk, R = HostStaging::kSlots * C;
  {
    HostStaging st;
    if (c == "sizes") {
      for (int delay : {0, 200})
        for (uint64_t n : {uint64_t(1), C - 1, C, C + 1, 4 * M, R - 1, R, R + 1, 3 * R + 12345, 2 * R}) {
          g_delayUs = delay;
          roundTrip(st, {n});
          roundTrip(st, {n, C / 2 + 3, n + 7});
        }
      need(g_pinned == 1 && g_events == static_cast<int>(HostStaging::kSlots), "one ring, one event per slot");
    } else if (c == "no_page_locked_memory") {
      g_failPinned = 1;
      need(!st.ready() && g_pinned == 0 && g_events == 0, "ready without memory");
      g_failPinned = 0;
      roundTrip(st, {5 * M});
    } else if (c == "no_events") {
      g_failEvents = 1;
      need(!st.ready() && g_pinned == 0 && g_events == 0, "ready without events");
      g_failEvents = 0;
      roundTrip(st, {5 * M});
    } else if (c == "failed_transfer") {
      for (int at : {0, 1, static_cast<int>(HostStaging::kSlots), 3 * static_cast<int>(HostStaging::kSlots) - 1}) {
        need(st.ready(), "ready");
        std::vector<uint8_t> host = bytes(3 * R), device(3 * R);
        for (bool down : {false, true}) {
          g_delayUs = 300;
          g_failCopy = at;
          bool threw = false;
          try {
            if (down) st.download(host.data(), device.data(), host.size(), nullptr);
            else st.upload(device.data(), host.data(), host.size(), nullptr);
          } catch (const denox::Error &) { threw = true; }
          need(threw, "an error of the link is reported");
          g_failCopy = -1;
          roundTrip(st, {2 * R + 5});
        }
      }
    } else if (c == "no_memory_for_threads") {
      need(st.ready(), "ready");
      std::vector<uint8_t> host = bytes(3 * R + 1), device(3 * R + 1), back(3 * R + 1);
      // whichever allocation is the first to fail, the call throws bad_alloc or does the work; it never ends the process
      for (bool down : {false, true})
        for (long at = 0; at < 40; ++at) {
          (void)hipStreamSynchronize(nullptr);
          std::fill(back.begin(), back.end(), uint8_t(0));
          std::memcpy(device.data(), host.data(), host.size());
          bool threw = false;
          g_failNew = at;
          try {
            // (the stand-in's own queue allocates as well: a failure there surfaces as one of the call's)
            if (down) st.download(back.data(), device.data(), back.size(), nullptr);
            else st.upload(device.data(), host.data(), host.size(), nullptr);
          } catch (const std::bad_alloc &) { threw = true; }
          g_failNew = -1;
          (void)hipStreamSynchronize(nullptr);
          if (down && !threw) need(back == host, "wrong bytes after a failed thread");
          if (!down && !threw) need(device == host, "wrong bytes after a failed thread");
        }
      roundTrip(st, {5 * M});
    } else need(false, "no such case");
  }
  need(g_pinned == 0 && g_events == 0, "memory or events left behind");
  push(nullptr);
  worker.join();
  std::printf("ok\n");
  return 0;
}
