// Host copies by several threads (runtime/host_copy.cpp) on their own: when the threads are started, and what happens where
// the system refuses them.  Built with shim.cpp by tests/test_host_copy_cpu.py.  Argument: how many threads are granted.
#include <dirent.h>
#include <dlfcn.h>
#include <pthread.h>

#include <cerrno>
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "../../i_amd/csrc/runtime/host_copy.h"

static int granted = 0;
extern "C" int pthread_create(pthread_t* thread, const pthread_attr_t* attr, void* (*run)(void*), void* arg) {
  if (granted-- <= 0) return EAGAIN;
  static auto real = reinterpret_cast<int (*)(pthread_t*, const pthread_attr_t*, void* (*)(void*), void*)>(dlsym(RTLD_NEXT, "pthread_create"));
  return real(thread, attr, run, arg);
}

namespace ihip {  // (hip_rt.cpp's part of it: nothing here transfers)
Err check(hipError_t e, const char* what) { return e == hipSuccess ? Err{} : Err(what); }
Err h2d(void*, const void*, size_t, hipStream_t) { return "not here"; }
Err d2h(void*, const void*, size_t, hipStream_t) { return "not here"; }
Err sync(hipStream_t) { return {}; }
}  // namespace ihip

static int threads() {
  int n = 0;
  DIR* d = opendir("/proc/self/task");
  while (dirent* e = readdir(d)) n += e->d_name[0] != '.';
  closedir(d);
  return n;
}

int main(int, char** argv) {
  const int asked = granted = std::atoi(argv[1]);
  std::vector<unsigned> from(3 << 20), to(from.size());
  for (size_t i = 0; i < from.size(); ++i) from[i] = (unsigned)(i * 2654435761u);
  {  // small copies: the caller alone
    ihip::copy_by_threads(to.data(), from.data(), 100);
    ihip::CopyAhead ahead({{to.data() + 25, from.data() + 25, 1000}, {to.data() + 275, from.data() + 275, 4}, {nullptr, nullptr, 0}});
    for (size_t n = 3; n-- > 0;) ahead.wait(n);
  }
  if (threads() != 1 || granted != asked) return std::puts("threads for a small copy"), 1;
  for (int round = 0; round < 20; ++round) {
    std::fill(to.begin(), to.end(), 0u);
    std::vector<ihip::CopyPiece> pieces;
    for (size_t at = 0; at < from.size(); at += 200003) pieces.push_back({&to[at], &from[at], 4 * std::min<size_t>(200003, from.size() - at)});
    ihip::CopyAhead ahead(pieces);
    for (size_t n = 0; n < pieces.size(); ++n) {
      ahead.wait(n);
      const size_t last = 200003 * n + pieces[n].bytes / 4 - 1;
      if (to[200003 * n] != from[200003 * n] || to[last] != from[last]) return std::puts("a piece that is not there"), 1;
    }
    if (to != from) return std::puts("wrong elements"), 1;
  }
  std::fill(to.begin(), to.end(), 0u);
  ihip::copy_by_threads(to.data(), from.data(), 4 * from.size());
  if (to != from) return std::puts("wrong elements of a block"), 1;
  if (threads() > 1 + asked) return std::puts("more threads than granted"), 1;
  std::printf("ok, %d threads\n", threads());
  std::fflush(stdout);
  std::_Exit(0);
}
