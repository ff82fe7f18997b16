// Host check of the copies between device ranges and the caller's arrays
// (staged_copy, uq_amd/csrc/lbm_io.hip), with the runtime's copy and allocation
// calls defined here over plain memory: with pinned slots, without any, with some
// of them refused, and where threads cannot be made (pthread_create fails, or the
// thread's own memory). Each copy must bring every byte and touch no other,
// segments of null left out, and keep the pool within its bound. Exits 1 on the
// first failure.
#include <atomic>
#include <cerrno>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <new>

#include <dlfcn.h>
#include <pthread.h>

#include "../uq_amd/csrc/lbm_io.hip"

static std::atomic<int> g_pinned_left{1 << 30}, g_slots{0};
static std::atomic<bool> g_no_threads{false}, g_no_memory{false};
static thread_local bool t_caller = false;

extern "C" hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
  if (g_pinned_left.fetch_sub(1) <= 0) return hipErrorOutOfMemory;
  g_slots++;
  *p = std::malloc(n);
  return hipSuccess;
}
extern "C" hipError_t hipHostFree(void* p) {
  g_slots--;
  std::free(p);
  return hipSuccess;
}
extern "C" hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
  *s = (hipStream_t)(size_t)16;
  return hipSuccess;
}
extern "C" hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
extern "C" hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
extern "C" hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
  std::memcpy(d, s, n);
  return hipSuccess;
}
extern "C" hipError_t hipGetDevice(int* d) {
  *d = 0;
  return hipSuccess;
}
extern "C" hipError_t hipSetDevice(int) { return hipSuccess; }
extern "C" hipError_t hipGetLastError(void) { return hipSuccess; }

// what std::thread calls
extern "C" int pthread_create(pthread_t* t, const pthread_attr_t* a, void* (*f)(void*), void* x) noexcept {
  using Create = int (*)(pthread_t*, const pthread_attr_t*, void* (*)(void*), void*);
  static const Create create = (Create)dlsym(RTLD_NEXT, "pthread_create");
  return g_no_threads ? EAGAIN : create(t, a, f, x);
}
void* operator new(size_t n) {
  // a copy's own lists are its first three allocations; what follows is the
  // threads' memory
  static thread_local int count = 0;
  if (!g_no_memory || !t_caller) count = 0;
  else if (++count > 3) throw std::bad_alloc();
  if (void* p = std::malloc(n ? n : 1)) return p;
  throw std::bad_alloc();
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, size_t) noexcept { std::free(p); }

static bool check(const char* what, size_t bytes, bool out) {
  // three segments of a device range, the middle one not wanted
  const size_t n[3] = {bytes / 3 + 1, bytes / 7 + 3, bytes - bytes / 3};
  std::vector<char> dev(n[0] + n[1] + n[2]), a(n[0] + 2, 0x55), c(n[2] + 2, 0x55);
  for (size_t k = 0; k < dev.size(); k++) dev[k] = (char)(k * 2654435761u >> 13);
  if (!out)
    for (size_t k = 0; k < a.size(); k++) a[k] = (char)(k * 40503u >> 5);
  if (!out)
    for (size_t k = 0; k < c.size(); k++) c[k] = (char)(k * 9176u >> 3);
  const std::vector<char> dev0 = dev, a0 = a, c0 = c;
  const std::vector<uqlbm::HostSeg> segs{{a.data() + 1, n[0]}, {nullptr, n[1]}, {c.data() + 1, n[2]}};
  t_caller = true;
  const hipError_t e = uqlbm::staged_copy(dev.data(), segs, out, nullptr);
  t_caller = false;
  bool ok = e == hipSuccess;
  std::vector<char> want_dev = dev0, want_a = a0, want_c = c0;
  if (out) {
    std::memcpy(want_a.data() + 1, dev0.data(), n[0]);
    std::memcpy(want_c.data() + 1, dev0.data() + n[0] + n[1], n[2]);
  } else {
    std::memcpy(want_dev.data(), a0.data() + 1, n[0]);
    std::memcpy(want_dev.data() + n[0] + n[1], c0.data() + 1, n[2]);
    // the part of no host array may hold anything
    std::memcpy(dev.data() + n[0], want_dev.data() + n[0], n[1]);
  }
  ok = ok && dev == want_dev && a == want_a && c == want_c && g_slots <= 16;
  std::printf("%s, %s, %zu bytes: %s\n", what, out ? "out" : "in", dev.size(), ok ? "ok" : "WRONG");
  std::fflush(stdout);
  return ok;
}

int main() {
  const size_t sizes[] = {1, 1000, size_t(1) << 20, (size_t(2) << 20) + 1, (size_t(23) << 20) + 77};
  bool ok = true;
  for (size_t n : sizes)
    for (bool out : {true, false}) {
      g_pinned_left = 0;
      ok = ok && check("no pinned memory", n, out);
      g_pinned_left = 3;
      ok = ok && check("pinned memory for three", n, out);
      g_pinned_left = 1 << 30;
      ok = ok && check("pinned", n, out);
      g_no_threads = true;
      ok = ok && check("no threads", n, out);
      g_no_threads = false;
      g_no_memory = true;
      ok = ok && check("no memory for threads", n, out);
      g_no_memory = false;
      uqlbm::release_slots();
      ok = ok && g_slots == 0;
    }
  return ok ? 0 : 1;
}
