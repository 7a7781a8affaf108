// Runs the pinned-ring copy (gn_copy.h) on the host, with each kind of failure
// at every place it can come: a call returns or throws, leaves no thread
// behind, and the next call copies every byte.
#include <cstdio>
#include <dlfcn.h>
#include <new>
#include <numeric>
#include <pthread.h>

#include "../../gonano_amd/csrc/gn_copy.h"

static thread_local long new_left = 0;  // this thread's nth allocation fails
static std::atomic<long> thread_left{0};

void* operator new(std::size_t n) {
  if (new_left > 0 && --new_left == 0) throw std::bad_alloc();
  if (void* p = std::malloc(n ? n : 1)) return p;
  throw std::bad_alloc();
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, std::size_t) noexcept { std::free(p); }

extern "C" int pthread_create(pthread_t* t, const pthread_attr_t* a, void* (*f)(void*), void* x) {
  static auto real = (int (*)(pthread_t*, const pthread_attr_t*, void* (*)(void*), void*))dlsym(
      RTLD_NEXT, "pthread_create");
  if (thread_left.load() > 0 && thread_left.fetch_sub(1) == 1) return EAGAIN;
  return real(t, a, f, x);
}

namespace gn {
void set_last_error(const std::string&) {}
}  // namespace gn

using gn::HostCopy;

// sizes that cut pieces, pack several into one, and leave odd ends
static bool copy_ok(HostCopy& c, const std::vector<size_t>& sizes, bool* threw) {
  const size_t total = std::accumulate(sizes.begin(), sizes.end(), (size_t)0);
  std::vector<unsigned char> src(total), dst(total, 0);
  for (size_t i = 0; i < total; i++) src[i] = (unsigned char)(i * 2654435761u >> 13);
  std::vector<HostCopy::Seg> segs;
  size_t o = 0;
  for (size_t n : sizes) {
    segs.push_back({dst.data() + o, src.data() + o, n});
    o += n;
  }
  *threw = false;
  try {
    c.download(0, nullptr, segs);
  } catch (const std::exception&) {
    *threw = true;
  }
  new_left = 0;
  thread_left = 0;
  fail_copy.left = fail_wait.left = fail_device.left = 0;
  return *threw || std::memcmp(src.data(), dst.data(), total) == 0;
}

int main() {
  const size_t M = HostCopy::PIECE;
  const std::vector<std::vector<size_t>> cases = {
      {1}, {M}, {M + 1}, {M - 1, 3, 255, 257, 1024, 2 * M}, {5 * M + 17, 12, 40, 13 * M, 1},
      std::vector<size_t>(3000, 2000), {60 * M + 5}};
  for (const auto& sizes : cases) {
    HostCopy c;
    bool threw;
    for (int r = 0; r < 3; r++)
      if (!copy_ok(c, sizes, &threw) || threw) return std::printf("plain copy\n"), 1;
  }
  const std::vector<size_t> sizes = {9 * M + 100, 7, 5 * M, 2000};
  const char* names[] = {"allocation", "thread", "copy", "wait", "device"};
  for (int kind = 0; kind < 5; kind++) {
    HostCopy c;
    int errors = 0;
    for (long at = 1; at <= 60; at++) {
      bool threw;
      // the vectors of copy_ok allocate first: 2 buffers and the segments' growth
      if (kind == 0) new_left = at + 5;
      if (kind == 1) thread_left = at;
      if (kind == 2) fail_copy.left = at;
      if (kind == 3) fail_wait.left = at;
      if (kind == 4) fail_device.left = at;
      if (!copy_ok(c, sizes, &threw)) return std::printf("%s failure %ld\n", names[kind], at), 1;
      errors += threw;
      // a thread or a device that cannot be had only means fewer helpers
      if (threw && (kind == 1 || kind == 4)) return std::printf("%s error\n", names[kind]), 1;
      if (!copy_ok(c, sizes, &threw) || threw)
        return std::printf("copy after a %s failure %ld\n", names[kind], at), 1;
    }
    if ((kind == 0 || kind == 2 || kind == 3) && errors == 0)
      return std::printf("%s failures were not seen\n", names[kind]), 1;
  }
  std::printf("ok\n");
  return 0;
}
