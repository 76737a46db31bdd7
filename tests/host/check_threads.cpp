// Work shared by host threads (kmst_threads.hpp) where threads cannot be
// created, or there is no memory for them: pthread_create and operator new
// fail from a given call on.
#include <dlfcn.h>
#include <pthread.h>

#include <cerrno>
#include <cstdio>
#include <cstdlib>
#include <new>
#include <stdexcept>

#include "kmst_threads.hpp"

namespace {
std::atomic<long> threads_left{1 << 30}, news_left{1 << 30};
}

extern "C" int pthread_create(pthread_t* t, const pthread_attr_t* a, void* (*f)(void*), void* x) {
  using Fn = int (*)(pthread_t*, const pthread_attr_t*, void* (*)(void*), void*);
  static const Fn real = reinterpret_cast<Fn>(dlsym(RTLD_NEXT, "pthread_create"));
  return threads_left.fetch_sub(1) > 0 ? real(t, a, f, x) : EAGAIN;
}
void* operator new(std::size_t n) {
  if (news_left.fetch_sub(1) > 0)
    if (void* p = std::malloc(n)) return p;
  throw std::bad_alloc();
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, std::size_t) noexcept { std::free(p); }

int main() {
  constexpr std::uint64_t N = 100000;
  std::vector<int> done(N);
  int bad = 0;
  auto check = [&](unsigned threads, std::uint64_t block, long creations, long news) {
    std::fill(done.begin(), done.end(), 0);
    threads_left = creations;
    news_left = news;
    try {
      kmst::for_blocks(threads, N, block, [&](std::uint64_t a, std::uint64_t b) {
        for (std::uint64_t i = a; i < b; ++i) ++done[i];
      });
    } catch (...) {
      ++bad;
      std::printf("thrown: ");
    }
    threads_left = news_left = 1 << 30;
    std::uint64_t once = 0;
    for (int x : done) once += x == 1;
    if (once != N) {
      ++bad;
      std::printf("%u threads, blocks of %llu, %ld creations, %ld allocations: %llu of %llu items\n",
                  threads, (unsigned long long)block, creations, news, (unsigned long long)once,
                  (unsigned long long)N);
    }
  };
  for (unsigned threads : {1u, 2u, 6u, 8u})
    for (std::uint64_t block : {std::uint64_t{1}, std::uint64_t{16384}, N, 2 * N})
      for (long k = 0; k < 8; ++k) {
        check(threads, block, k, 1 << 30);
        check(threads, block, 1 << 30, k);
      }
  // a failure in the work comes out once all have ended
  for (long k : {0L, 3L, 100L}) {
    threads_left = k;
    bool thrown = false;
    try {
      kmst::on_threads(6, [](unsigned t) {
        if (t == 0) throw std::runtime_error("work");
      });
    } catch (const std::runtime_error&) {
      thrown = true;
    }
    bad += !thrown;
  }
  if (!bad) std::printf("ok (threads)\n");
  return bad != 0;
}
