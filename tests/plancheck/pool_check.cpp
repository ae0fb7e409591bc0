// Loops on the kept worker threads, from several threads at once: nested, with exceptions,
// while holders come and go, and in a forked child. Exit code 0: every loop did every item
// once, with a thread number below its thread count.
#include <sys/wait.h>
#include <unistd.h>

#include <cstdio>
#include <stdexcept>

#include "../../chemps2_amd/csrc/parallel.hpp"

using namespace chm;

static bool loop(int n, int threads) {
  std::vector<long> part(threads, 0);
  std::atomic<bool> bad{false};
  parallel_for(n, threads, [&](int64_t i, int tid) {
    if (tid < 0 || tid >= threads) bad = true;
    else part[tid] += i;
  });
  long sum = 0;
  for (long v : part) sum += v;
  return !bad && sum == (long)n * (n - 1) / 2;
}

int main() {
  for (int rep = 0; rep < 40; rep++) {
    Pool::Ref a;
    std::atomic<int> bad{0};
    std::vector<std::thread> callers;
    for (int q = 0; q < 4; q++)
      callers.emplace_back([&, q] {
        Pool::Ref c;
        for (int k = 0; k < 25; k++) {
          if (!loop(1 + (k * 37 + q) % 300, 1 + (k + q) % 16)) bad++;
          bool caught = false;
          try {
            parallel_for(100, 8, [&](int64_t i, int) { if (i == 50) throw std::runtime_error("item"); });
          } catch (const std::runtime_error&) {
            caught = true;
          }
          if (!caught) bad++;
          parallel_for(6, 4, [&](int64_t, int) { if (!loop(40, 3)) bad++; });
        }
      });
    for (auto& t : callers) t.join();
    if (bad) return std::printf("%d loops failed\n", bad.load()), 1;
  }
  for (int rep = 0; rep < 20; rep++) {
    Pool::Ref a;
    if (!loop(1000, 8)) return 2;
    const pid_t p = fork();
    if (p == 0) _exit(loop(1000, 8) ? 0 : 1);
    int st = 0;
    waitpid(p, &st, 0);
    if (st != 0) return 3;
  }
  return loop(1000, 8) ? 0 : 4;  // no holder any more
}
