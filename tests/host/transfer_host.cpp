// C entries over colphys::Transfer for tests/test_transfer_host.py.
#include "../../roundabout_amd/csrc/transfer.h"

#include <new>

#include <signal.h>
#include <sys/syscall.h>
#include <time.h>
#include <unistd.h>

// operator new of this library alone (linked -Bsymbolic)
static bool no_memory = false;
void* operator new(size_t n) {
  void* const p = no_memory ? nullptr : std::malloc(n ? n : 1);
  if (!p) throw std::bad_alloc();
  return p;
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, size_t) noexcept { std::free(p); }

static int hold_ms = 0;
static void hold(int) {
  timespec t{hold_ms / 1000, (hold_ms % 1000) * 1000000L};
  while (nanosleep(&t, &t) != 0) {
  }
}

extern "C" {

colphys::Transfer* tr_new() { return new colphys::Transfer; }
void tr_delete(colphys::Transfer* t) { delete t; }
HostStream* tr_stream() { return new HostStream; }
void tr_busy(HostStream* s, double seconds) {
  s->busy_until = std::chrono::steady_clock::now() + std::chrono::microseconds((long long)(1e6 * seconds));
}
int tr_to_host(colphys::Transfer* t, void* dst, const void* dev, size_t n, HostStream* s) {
  return t->to_host(dst, dev, n, s);
}
int tr_to_device(colphys::Transfer* t, void* dev, const void* src, size_t n, HostStream* s) {
  return t->to_device(dev, src, n, s);
}
int tr_sync(HostStream* s) { return hipStreamSynchronize(s); }
void tr_copy(colphys::Transfer* t, void* dst, const void* src, size_t n) { t->copy(dst, src, n); }
// thread `tid` of this process stands still for `ms`
void tr_hold(int tid, int ms) {
  hold_ms = ms;
  signal(SIGUSR2, hold);
  syscall(SYS_tgkill, getpid(), tid, SIGUSR2);
}
void tr_no_memory(int on) { no_memory = on != 0; }
void tr_refuse_pinned(int on) { g_hip.refuse_pinned = on != 0; }
int tr_last_error() { return hipGetLastError(); }

}  // extern "C"
