// transfer.hip -- see transfer.h.
#include "transfer.h"

#include <sched.h>

#include <algorithm>
#include <atomic>
#include <chrono>
#include <condition_variable>
#include <cstdint>
#include <cstring>
#include <exception>
#include <mutex>
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
constexpr int PIECES = 32;  // of a block that the threads copy
constexpr size_t WORTH = 512u << 10;  // bytes for which one more thread is woken

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
  // The threads copy a block at a time and are woken only when the bytes are
  // there: a wait for the stream (the work queued before the transfer, which
  // may take seconds) is the calling thread's alone.  A block is cut into
  // 32 pieces; each thread has a run of its own, the same one in every block
  // (its processor's caches and a huge page of a fresh destination), and goes
  // on to what others have not begun, so that one that is late or loses its
  // processor holds up no more than the piece it is at.
  std::mutex m;
  std::condition_variable cv, cv_done;
  std::vector<std::thread> threads;
  bool quit = false, caller_waits = false;
  int n_threads = 0;  // 0: not started
  int sleeping = 0;
  uint64_t calls = 0;  // bumped by call_up
  // the block's number in the high half, a bit for each piece not yet taken in
  // the low one: nothing is taken of a block that is done, whatever came after
  std::atomic<uint64_t> open{0};
  std::atomic<int> left{0};  // pieces not yet copied; at 0 the next block may be set up
  char* dst = nullptr;
  const char* src = nullptr;
  size_t bytes = 0, piece = 0;
  // pinned chunks, made at the first transfer that needs them
  char* slot[NSLOT] = {nullptr, nullptr, nullptr, nullptr};
  hipEvent_t done[NSLOT] = {nullptr, nullptr, nullptr, nullptr};
  size_t slot_bytes = 0;

  static size_t chunk_of(size_t n) { return n >= BIG ? BIG_CHUNK : SMALL_CHUNK; }

  // the pieces that are thread t's own (the caller is thread 0 of n)
  static uint32_t own_of(int t, int n) {
    const int a = PIECES * t / n, b = PIECES * (t + 1) / n;
    return (uint32_t)((1ull << b) - (1ull << a));
  }
  // take a piece, of `own` before others', and copy it; false if there is none
  bool take(uint32_t own) {
    uint64_t o = open.load(std::memory_order_acquire);
    int k;
    do {
      const uint32_t mine = (uint32_t)o & own;
      if ((uint32_t)o == 0) return false;
      k = mine ? __builtin_ctz(mine) : 31 - __builtin_clz((uint32_t)o);
    } while (!open.compare_exchange_weak(o, o & ~(1ull << k), std::memory_order_acq_rel, std::memory_order_acquire));
    const size_t at = piece * (size_t)k;
    std::memcpy(dst + at, src + at, std::min(piece, bytes - at));
    if (left.fetch_sub(1, std::memory_order_acq_rel) == 1) {
      std::lock_guard<std::mutex> lk(m);
      if (caller_waits) cv_done.notify_one();
    }
    return true;
  }
  bool some() const { return (uint32_t)open.load(std::memory_order_acquire) != 0; }

  void work(int t, int n) {
    const uint32_t own = own_of(t, n);
    uint64_t heard = 0;
    for (;;) {
      while (take(own)) {
      }
      if (spin_for([&] { return some(); })) continue;
      std::unique_lock<std::mutex> lk(m);
      ++sleeping;
      cv.wait(lk, [&] { return quit || some() || calls != heard; });
      --sleeping;
      heard = calls;
      if (quit) return;
    }
  }

  // Wake as many threads as `n` bytes are worth: a wake-up costs the thread
  // some tens of microseconds, and the caller some of its own for each call.
  void wake(size_t n, bool ahead = false) {
    std::lock_guard<std::mutex> lk(m);
    if (ahead) ++calls;
    if (sleeping == 0) return;
    const size_t want = n / WORTH;
    if (2 * want >= (size_t)sleeping)
      cv.notify_all();
    else
      for (size_t i = 0; i < want; ++i) cv.notify_one();
  }

  // A chunk of `n` bytes may be here soon: the threads' way out of their sleep
  // overlaps its transfer.  (If it is not, they are back asleep in 50 us.)
  void call_up(size_t n) { wake(n, true); }

  // A block, copied by the threads and the caller; returns when it is.
  void share(void* d, const void* s, size_t n) {
    dst = (char*)d;
    src = (const char*)s;
    bytes = n;
    piece = (n / PIECES + 4096) / 4096 * 4096;
    const int pieces = (int)((n + piece - 1) / piece);
    left.store(pieces, std::memory_order_relaxed);
    const uint64_t number = (open.load(std::memory_order_relaxed) >> 32) + 1;
    open.store(number << 32 | ((1ull << pieces) - 1), std::memory_order_release);
    wake(n);
    const uint32_t own = own_of(0, n_threads);
    while (take(own)) {
    }
    if (!spin_for([&] { return left.load(std::memory_order_acquire) == 0; })) {
      std::unique_lock<std::mutex> lk(m);
      caller_waits = true;
      cv_done.wait(lk, [&] { return left.load(std::memory_order_acquire) == 0; });
      caller_waits = false;
    }
  }

  void start() {
    if (n_threads > 0) return;
    const int want = std::max(1, std::min(MAX_THREADS, allowed_cpus() / 2));
    try {
      for (int t = 1; t < want; ++t) threads.emplace_back([this, t, want] { work(t, want); });
    } catch (const std::exception&) {
      // no thread or no memory for one, and the callers are C: fewer threads than wanted: those there are do the work
    }
    n_threads = want;  // (the shares of threads that are not there are taken by the others)
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
  // Whether a transfer of `n` bytes goes through the chunks.  Where they are
  // not to be had it does not, and that is no error: what the failed call
  // left for hipGetLastError goes with it, or the next launch's check would
  // find it.
  bool takes(size_t n) {
    if (n < SMALL) return false;
    if (prepare(n) == hipSuccess) return true;
    (void)hipGetLastError();
    return false;
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
  hipError_t e = hipSuccess;
  if (!im.takes(bytes)) {
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
  im.call_up(std::min(chunk, bytes));
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
  hipError_t e = hipSuccess;
  if (!im.takes(bytes)) {
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
  for (size_t at = 0; at < bytes; at += BIG)
    im.share((char*)dst + at, (const char*)src + at, std::min(BIG, bytes - at));
}

}  // namespace colphys
