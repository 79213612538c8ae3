// transfer.cpp — matrix elements to the device through pinned buffers.
#include "transfer.hpp"

#include <algorithm>
#include <atomic>
#include <exception>
#include <mutex>
#include <thread>
#include <vector>

#include "internal.hpp"

namespace mlem {

namespace {

// Chunks of 2 MB: a pinned buffer that stays in the CPU's caches between the
// memcpy and the copy engine, and few pages to map. Two 64 MB buffers filled by
// one thread loaded 372 MB in 61 ms, this takes 12 (55 GB/s is the link's 7).
constexpr uint64_t kChunk = 2ull << 20;
constexpr uint64_t kParallelBytes = 16ull << 20;  // threads pay off above this
constexpr int kThreads = 4;                       // memcpy 30 -> 81 GB/s; the link takes 55

}  // namespace

void stream_to_device(void* dst, uint64_t bytes, int device, hipStream_t s,
                      const Produce& produce) {
  if (bytes == 0) return;
  const int hw = (int)std::max(1u, std::thread::hardware_concurrency());
  const int nt = bytes < kParallelBytes ? 1 : std::min(kThreads, hw);
  struct Pinned {
    char* p = nullptr;
    std::vector<hipEvent_t> ev;
    ~Pinned() {
      for (hipEvent_t e : ev) (void)hipEventDestroy(e);
      if (p) (void)hipHostFree(p);
    }
  } pin;
  const uint64_t chunk = std::min(kChunk, bytes);
  MLEM_HIP(hipHostMalloc((void**)&pin.p, chunk * 2 * nt, hipHostMallocDefault));
  for (int i = 0; i < 2 * nt; ++i) {
    hipEvent_t e;
    MLEM_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
    pin.ev.push_back(e);
  }
  std::atomic<uint64_t> next{0};
  std::atomic<bool> stop{false};
  std::exception_ptr error;
  std::mutex mu;
  char* d = static_cast<char*>(dst);
  auto work = [&](int t) {
    try {
      if (t) MLEM_HIP(hipSetDevice(device));
      bool used[2] = {false, false};
      for (int b = 0; !stop; b ^= 1) {
        const uint64_t off = next.fetch_add(chunk);
        if (off >= bytes) break;
        const uint64_t n = std::min(chunk, bytes - off);
        char* buf = pin.p + chunk * (2 * t + b);
        hipEvent_t e = pin.ev[(size_t)(2 * t + b)];
        if (used[b]) MLEM_HIP(hipEventSynchronize(e));
        produce(buf, off, n);
        MLEM_HIP(hipMemcpyAsync(d + off, buf, n, hipMemcpyHostToDevice, s));
        MLEM_HIP(hipEventRecord(e, s));
        used[b] = true;
      }
    } catch (...) {
      stop = true;
      std::lock_guard<std::mutex> lock(mu);
      if (!error) error = std::current_exception();
    }
  };
  std::vector<std::thread> pool;
  try {
    for (int t = 1; t < nt; ++t) pool.emplace_back(work, t);
  } catch (...) {  // no more threads: the ones there do the work
  }
  work(0);
  for (std::thread& th : pool) th.join();
  const hipError_t e = hipStreamSynchronize(s);  // the buffers are free, also after an error
  if (error) std::rethrow_exception(error);
  MLEM_HIP(e);
}

}  // namespace mlem
