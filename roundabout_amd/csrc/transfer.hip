// transfer.hip -- see transfer.h.
#include "transfer.h"

#include <sched.h>

#include <algorithm>
#include <atomic>
#include <chrono>
#include <condition_variable>
#include <cstdint>
#include <cstring>
#include <mutex>
#include <system_error>
#include <thread>
#include <vector>

namespace colphys {

namespace {

constexpr int NSLOT = 4;
constexpr int MAX_THREADS = 8;  // the caller and seven more
// Below this size the runtime's own copy is taken: at 0.66 MB the two are
// equal (0.04 ms up, 0.055 ms down), at 1.6 MB this one takes 0.06 and 0.08
// ms instead of 0.08 and 0.11.
constexpr size_t SMALL = 1u << 20;
// Chunks: small ones overlap copy and transfer in a transfer of a few MB;
// in a large one each of eight threads fills 2 MiB, a huge page of a fresh
// destination, to itself.  104 MB up: 3.8 ms by the runtime, 2.3 in chunks of
// 4 MiB, 2.0 of 16 (52 GB/s, the link's rate); down into a fresh array 6.1
// (10 at worst), 4.6, 2.3 to 3.0.
constexpr size_t SMALL_CHUNK = 4u << 20, BIG_CHUNK = 16u << 20, BIG = 64u << 20;

int allowed_cpus() {
  cpu_set_t set;
  CPU_ZERO(&set);
  return sched_getaffinity(0, sizeof set, &set) == 0 ? CPU_COUNT(&set) : 1;
}

// A short wait for a condition that another running thread is about to set:
// tens of microseconds, then the caller sleeps on a condition variable.
template <class Cond>
bool spin_for(Cond cond) {
  constexpr auto SPIN = std::chrono::microseconds(50);
  const auto end = std::chrono::steady_clock::now() + SPIN;
  for (int i = 0;; ++i) {
    if (cond()) return true;
    if (i % 16 == 15 && std::chrono::steady_clock::now() > end) return false;
  }
}

}  // namespace

struct Transfer::Impl {
  std::mutex call;  // one transfer at a time
  // The threads copy a block at a time, each its part, and are woken only
  // when the bytes are there: a wait for the stream (the work queued before
  // the transfer, which may take seconds) is the calling thread's alone.
  std::mutex m;
  std::condition_variable cv, cv_done;
  std::vector<std::thread> threads;
  int n_threads = 0;  // 0: not started
  int sleeping = 0;
  bool quit = false;
  std::atomic<uint64_t> turn{0};  // bumped for each block
  std::atomic<int> left{0};       // threads still on it
  char* dst = nullptr;
  const char* src = nullptr;
  size_t bytes = 0;
  // pinned chunks, made at the first transfer that needs them
  char* slot[NSLOT] = {nullptr, nullptr, nullptr, nullptr};
  hipEvent_t done[NSLOT] = {nullptr, nullptr, nullptr, nullptr};
  size_t slot_bytes = 0;

  static size_t chunk_of(size_t n) { return n >= BIG ? BIG_CHUNK : SMALL_CHUNK; }

  // part `t` of the block, in whole pages of 4 KiB where it can be
  void part(int t) {
    const size_t per = (bytes / (size_t)n_threads + 4095) / 4096 * 4096;
    const size_t a = std::min(bytes, per * (size_t)t), b = t + 1 == n_threads ? bytes : std::min(bytes, per * (size_t)(t + 1));
    if (b > a) std::memcpy(dst + a, src + a, b - a);
    if (left.fetch_sub(1, std::memory_order_acq_rel) == 1) {
      std::lock_guard<std::mutex> lk(m);
      cv_done.notify_one();
    }
  }

  void work(int t) {
    uint64_t seen = 0;
    for (;;) {
      if (!spin_for([&] { return turn.load(std::memory_order_acquire) != seen; })) {
        std::unique_lock<std::mutex> lk(m);
        ++sleeping;
        cv.wait(lk, [&] { return quit || turn.load(std::memory_order_acquire) != seen; });
        --sleeping;
        if (quit) return;
      }
      ++seen;  // (the caller waits for every thread before the next turn)
      part(t);
    }
  }

  // A block, copied by the threads and the caller; returns when it is.
  void share(void* d, const void* s, size_t n) {
    dst = (char*)d;
    src = (const char*)s;
    bytes = n;
    left.store(n_threads, std::memory_order_relaxed);
    turn.fetch_add(1, std::memory_order_release);
    {
      std::lock_guard<std::mutex> lk(m);
      if (sleeping > 0) cv.notify_all();
    }
    part(0);
    if (!spin_for([&] { return left.load(std::memory_order_acquire) == 0; })) {
      std::unique_lock<std::mutex> lk(m);
      cv_done.wait(lk, [&] { return left.load(std::memory_order_acquire) == 0; });
    }
  }

  void start() {
    if (n_threads > 0) return;
    const int want = std::max(1, std::min(MAX_THREADS, allowed_cpus() / 2));
    try {
      for (int t = 1; t < want; ++t) threads.emplace_back([this, t] { work(t); });
    } catch (const std::system_error&) {
      // fewer threads than wanted: those there are do the work
    }
    n_threads = (int)threads.size() + 1;
  }
  hipError_t prepare(size_t n) {
    start();
    const size_t need = chunk_of(n);
    if (slot_bytes >= need) return hipSuccess;
    for (int q = 0; q < NSLOT; ++q) {
      hipError_t e = done[q] ? hipEventSynchronize(done[q])  // a transfer may still read the slot
                             : hipEventCreateWithFlags(&done[q], hipEventDisableTiming);
      if (e != hipSuccess) return e;
    }
    slot_bytes = 0;
    for (int q = 0; q < NSLOT; ++q) {
      if (slot[q]) (void)hipHostFree(slot[q]);
      slot[q] = nullptr;
      const hipError_t e = hipHostMalloc((void**)&slot[q], need, hipHostMallocDefault);
      if (e != hipSuccess) {
        slot[q] = nullptr;
        return e;
      }
    }
    slot_bytes = need;
    return hipSuccess;
  }
};

Transfer::Transfer() : im_(new Impl) {}

Transfer::~Transfer() {
  {
    std::lock_guard<std::mutex> lk(im_->m);
    im_->quit = true;
    im_->cv.notify_all();
  }
  for (std::thread& t : im_->threads) t.join();
  for (int q = 0; q < NSLOT; ++q) {
    if (im_->done[q]) {
      (void)hipEventSynchronize(im_->done[q]);
      (void)hipEventDestroy(im_->done[q]);
    }
    if (im_->slot[q]) (void)hipHostFree(im_->slot[q]);
  }
}

hipError_t Transfer::to_host(void* dst, const void* dev, size_t bytes, hipStream_t stream) {
  Impl& im = *im_;
  std::lock_guard<std::mutex> lk(im.call);
  hipError_t e = bytes < SMALL ? hipSuccess : im.prepare(bytes);
  if (bytes < SMALL || e != hipSuccess) {
    e = hipMemcpyAsync(dst, dev, bytes, hipMemcpyDeviceToHost, stream);
    return e == hipSuccess ? hipStreamSynchronize(stream) : e;
  }
  const size_t chunk = Impl::chunk_of(bytes), n = (bytes + chunk - 1) / chunk;
  auto fetch = [&](size_t i) {
    const size_t at = i * chunk;
    hipError_t r = hipMemcpyAsync(im.slot[i % NSLOT], (const char*)dev + at, std::min(chunk, bytes - at),
                                  hipMemcpyDeviceToHost, stream);
    return r == hipSuccess ? hipEventRecord(im.done[i % NSLOT], stream) : r;
  };
  size_t sent = 0;
  for (; sent < std::min<size_t>(n, NSLOT) && e == hipSuccess; ++sent) e = fetch(sent);
  for (size_t i = 0; i < n && e == hipSuccess; ++i) {
    e = hipEventSynchronize(im.done[i % NSLOT]);
    if (e != hipSuccess) break;
    const size_t at = i * chunk;
    im.share((char*)dst + at, im.slot[i % NSLOT], std::min(chunk, bytes - at));
    if (sent < n) e = fetch(sent++);
  }
  return e;
}

hipError_t Transfer::to_device(void* dev, const void* src, size_t bytes, hipStream_t stream) {
  Impl& im = *im_;
  std::lock_guard<std::mutex> lk(im.call);
  hipError_t e = bytes < SMALL ? hipSuccess : im.prepare(bytes);
  if (bytes < SMALL || e != hipSuccess) {
    e = hipMemcpyAsync(dev, src, bytes, hipMemcpyHostToDevice, stream);
    return e == hipSuccess ? hipStreamSynchronize(stream) : e;
  }
  const size_t chunk = Impl::chunk_of(bytes), n = (bytes + chunk - 1) / chunk;
  for (size_t i = 0; i < n && e == hipSuccess; ++i) {
    // the slot's last transfer, of this call or an earlier one
    e = hipEventSynchronize(im.done[i % NSLOT]);
    if (e != hipSuccess) break;
    const size_t at = i * chunk, len = std::min(chunk, bytes - at);
    im.share(im.slot[i % NSLOT], (const char*)src + at, len);
    e = hipMemcpyAsync((char*)dev + at, im.slot[i % NSLOT], len, hipMemcpyHostToDevice, stream);
    if (e == hipSuccess) e = hipEventRecord(im.done[i % NSLOT], stream);
  }
  return e;
}

void Transfer::copy(void* dst, const void* src, size_t bytes) {
  Impl& im = *im_;
  if (bytes < SMALL) {
    std::memcpy(dst, src, bytes);
    return;
  }
  std::lock_guard<std::mutex> lk(im.call);
  im.start();
  im.share(dst, src, bytes);
}

}  // namespace colphys
