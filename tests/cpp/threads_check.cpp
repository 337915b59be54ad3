// threads_check.cpp — work over host threads where the system refuses some or all of them
// (runtime.hpp, parallel_for). The program's own pthread_create stands in for the system's.
#include <dlfcn.h>
#include <errno.h>
#include <pthread.h>

#include <cstdio>

#include "runtime.hpp"

static int allowed = 0;

extern "C" int pthread_create(pthread_t* t, const pthread_attr_t* a, void* (*f)(void*), void* arg) {
  if (allowed == 0) return EAGAIN;
  --allowed;
  using Fn = int (*)(pthread_t*, const pthread_attr_t*, void* (*)(void*), void*);
  return ((Fn)dlsym(RTLD_NEXT, "pthread_create"))(t, a, f, arg);
}

int main() {
  for (int threads : {0, 1, 2, 100}) {
    allowed = threads;
    std::vector<int> done(1000, 0);
    qr::parallel_for(done.size(), [&](uint64_t i) { done[i]++; });
    for (int d : done)
      if (d != 1) {
        std::printf("FAIL: work left out or done twice with %d threads\n", threads);
        return 1;
      }
    allowed = threads;
    bool caught = false;
    try {
      qr::parallel_for(100, [&](uint64_t i) {
        if (i >= 40) throw qr::Error{QR_ERR_ARG, std::to_string(i)};
      });
    } catch (const qr::Error& e) {
      caught = e.msg == "40";
    }
    if (!caught) {
      std::printf("FAIL: the lowest error with %d threads\n", threads);
      return 1;
    }
  }
  std::printf("ok\n");
  return 0;
}
