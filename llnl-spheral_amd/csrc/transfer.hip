// The calls that hand fields over: the isotropy test of an uploaded H, derivative
// fields from slot order to the caller's order, and large downloads.
#include "internal.hh"
#include "dgeom.hh"

#include <atomic>
#include <condition_variable>
#include <cstring>
#include <mutex>
#include <system_error>
#include <thread>

namespace sphgpu {

namespace {

// Bound by reading H once (101 MB at 2.1 M rows in 3-D: 0.04 ms; the host loop
// took 8 ms there).  A workgroup that meets a row of another form stores to the
// caller's word; which one does so last makes no difference.
template <int D>
__global__ void __launch_bounds__(256) k_not_isotropic(const double* __restrict__ H, int64_t n, int32_t* flag) {
  constexpr int NS = NSym<D>::value;
  const int64_t i = blockIdx.x * int64_t(256) + threadIdx.x;
  bool iso = true;
  if (i < n) {
    const double* h = H + i * NS;
    int k = 0;
    for (int a = 0; a < D; ++a)
      for (int b = a; b < D; ++b, ++k) iso = iso && (a == b ? h[k] == h[0] : h[k] == 0.0);
  }
  if (!iso) *flag = 1;
}

// One lane per value: the writes and, since slots follow the caller's nodes in
// runs, most reads are whole lines: 0.01 ms for 9 doubles of 125 k nodes, far
// below the copy that follows.
__global__ void __launch_bounds__(256) k_unsort(const double* __restrict__ src, const int32_t* __restrict__ iperm,
                                                int64_t values, int comps, double* __restrict__ dst) {
  const int64_t q = blockIdx.x * int64_t(256) + threadIdx.x;
  if (q >= values) return;
  const int64_t i = q / comps;
  dst[q] = src[int64_t(iperm[i]) * comps + (q - i * comps)];
}

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

}  // namespace

void copyToHost(Sim& s, void* host, const void* dev, size_t bytes) {
  auto plain = [&] {
    if (bytes) SG_CHECK_HIP(hipMemcpyAsync(host, dev, bytes, hipMemcpyDeviceToHost, s.stream));
    SG_CHECK_HIP(hipStreamSynchronize(s.stream));
  };
  if (bytes < kRingFrom) return plain();
  while (int(s.ringDone.size()) < kRingSlots) {
    hipEvent_t e;
    SG_CHECK_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
    s.ringDone.push_back(e);
  }
  if (!s.ring) SG_CHECK_HIP(hipHostMalloc(&s.ring, kRingSlot * kRingSlots, hipHostMallocDefault));
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

int32_t* queueIsotropyTest(Sim& s, const double* H, int64_t rows) {
  int32_t* flag = static_cast<int32_t*>(hostStaging(s, 0, sizeof(int32_t)));
  *flag = 0;
  const dim3 grid(unsigned((rows + 255) / 256));
  if (s.dim == 1) hipLaunchKernelGGL(k_not_isotropic<1>, grid, dim3(256), 0, s.stream, H, rows, flag);
  else if (s.dim == 2) hipLaunchKernelGGL(k_not_isotropic<2>, grid, dim3(256), 0, s.stream, H, rows, flag);
  else hipLaunchKernelGGL(k_not_isotropic<3>, grid, dim3(256), 0, s.stream, H, rows, flag);
  SG_CHECK_HIP(hipGetLastError());
  return flag;
}

const double* unsortDerivative(Sim& s, const double* src, int comps) {
  const int64_t values = s.nInt * comps;
  s.unsorted.ensure(sizeof(double) * size_t(values));
  hipLaunchKernelGGL(k_unsort, dim3(unsigned((values + 255) / 256)), dim3(256), 0, s.stream, src,
                     s.iperm.as<int32_t>(), values, comps, s.unsorted.as<double>());
  SG_CHECK_HIP(hipGetLastError());
  return s.unsorted.as<double>();
}

}  // namespace sphgpu
