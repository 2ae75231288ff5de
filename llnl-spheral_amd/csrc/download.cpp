// Downloads (host code).
#include "internal.hh"

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstring>
#include <mutex>
#include <system_error>
#include <thread>

namespace sphgpu {

namespace {

// Large downloads.  A caller's array is often fresh memory, and one thread that
// faults its pages in takes 24 ms for 100 MB, four times the transfer; the runtime's
// own staging is that one thread.  So the copy goes through pinned slots: this thread
// starts the transfers in order and several take the chunks that have landed to
// their place.  8 MB of slots keep the transfer going while eight threads
// work; below kRingFrom starting them costs what they save.  State of 2.1 M nodes
// (235 MB): 22.8 -> 10.1 ms.
constexpr size_t kRingSlot = size_t(1) << 20, kRingFrom = size_t(4) << 20;
constexpr int kRingSlots = 8, kRingThreads = 8;

struct RingCopy {
  const char* ring;
  char* host;
  size_t bytes;
  int64_t chunks;
  std::mutex m;
  std::condition_variable landedCv, freeCv;
  int64_t landed = 0;               // chunks in their slots, in order
  std::vector<char> taken;          // chunks copied out
  std::atomic<int64_t> next{0};
  bool stop = false;
  std::vector<std::thread> threads;

  RingCopy(const void* r, void* h, size_t b)
      : ring(static_cast<const char*>(r)), host(static_cast<char*>(h)), bytes(b),
        chunks(int64_t((b + kRingSlot - 1) / kRingSlot)), taken(size_t(chunks), 0) {}
  size_t size(int64_t c) const { return std::min(kRingSlot, bytes - size_t(c) * kRingSlot); }
  void work() {
    for (;;) {
      const int64_t c = next++;
      if (c >= chunks) return;
      {
        std::unique_lock<std::mutex> l(m);
        landedCv.wait(l, [&] { return stop || landed > c; });
        if (stop) return;
      }
      std::memcpy(host + size_t(c) * kRingSlot, ring + size_t(c % kRingSlots) * kRingSlot, size(c));
      {
        std::lock_guard<std::mutex> l(m);
        taken[size_t(c)] = 1;
      }
      freeCv.notify_one();
    }
  }
  // as many threads as the system gives; none: false
  bool start() {
    try {
      const int want = int(std::min<int64_t>(kRingThreads, chunks / 2));
      threads.reserve(size_t(want));
      for (int q = 0; q < want; ++q) threads.emplace_back([this] { work(); });
    } catch (const std::system_error&) {
    }
    return !threads.empty();
  }
  ~RingCopy() {
    {
      std::lock_guard<std::mutex> l(m);
      stop = stop || landed < chunks;
    }
    landedCv.notify_all();
    for (auto& t : threads) t.join();
  }
};

// The slots and their events; false where the system has none to give.
bool ringSlots(Sim& s) {
  auto got = [](hipError_t e) {
    if (e != hipSuccess) (void)hipGetLastError();   // handled here: not the next call's
    return e == hipSuccess;
  };
  while (int(s.ringDone.size()) < kRingSlots) {
    hipEvent_t e;
    if (!got(hipEventCreateWithFlags(&e, hipEventDisableTiming))) return false;
    s.ringDone.push_back(e);
  }
  if (!s.ring && !got(hipHostMalloc(&s.ring, kRingSlot * kRingSlots, hipHostMallocDefault))) s.ring = nullptr;
  return s.ring != nullptr;
}

}  // namespace

void copyToHost(Sim& s, void* host, const void* dev, size_t bytes) {
  auto plain = [&] {
    if (bytes) SG_CHECK_HIP(hipMemcpyAsync(host, dev, bytes, hipMemcpyDeviceToHost, s.stream));
    SG_CHECK_HIP(hipStreamSynchronize(s.stream));
  };
  if (bytes < kRingFrom || !ringSlots(s)) return plain();
  RingCopy r(s.ring, host, bytes);
  if (!r.start()) {
    r.landed = r.chunks;           // no thread waits
    return plain();
  }
  for (int64_t issued = 0, landed = 0; landed < r.chunks;) {
    // transfers into every slot that is free
    for (; issued < r.chunks; ++issued) {
      if (issued >= kRingSlots) {
        std::unique_lock<std::mutex> l(r.m);
        const size_t before = size_t(issued - kRingSlots);
        if (landed == issued) r.freeCv.wait(l, [&] { return r.taken[before] != 0; });
        else if (!r.taken[before]) break;
      }
      const size_t slot = size_t(issued % kRingSlots);
      SG_CHECK_HIP(hipMemcpyAsync(static_cast<char*>(s.ring) + slot * kRingSlot,
                                  static_cast<const char*>(dev) + size_t(issued) * kRingSlot, r.size(issued),
                                  hipMemcpyDeviceToHost, s.stream));
      SG_CHECK_HIP(hipEventRecord(s.ringDone[slot], s.stream));
    }
    SG_CHECK_HIP(hipEventSynchronize(s.ringDone[size_t(landed % kRingSlots)]));
    {
      std::lock_guard<std::mutex> l(r.m);
      r.landed = ++landed;
    }
    r.landedCv.notify_all();
  }
}                                  // joins: every chunk is in place

}  // namespace sphgpu
