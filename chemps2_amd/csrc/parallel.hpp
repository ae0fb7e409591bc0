// Host threads of the work-list generators: a dynamic loop over [0, n) that keeps the first
// exception and rethrows it on the calling thread.
#pragma once
#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstdint>
#include <cstdlib>
#include <exception>
#include <mutex>
#include <system_error>
#include <thread>
#include <vector>

#include <pthread.h>

namespace chm {

// CHM_THREADS, else OMP_NUM_THREADS, else the hardware's count; at most 64.
inline int host_threads() {
  for (const char* name : {"CHM_THREADS", "OMP_NUM_THREADS"}) {
    const char* v = std::getenv(name);
    if (v && std::atoi(v) > 0) return std::min(64, std::atoi(v));
  }
  const unsigned h = std::thread::hardware_concurrency();
  return (int)std::max(1u, std::min(64u, h));
}

// Worker threads kept while a holder lives (a library context holds a Pool::Ref): a step of a
// small sweep runs some fifty short loops, and starting and joining fifteen threads for each
// took longer than the loops. With the operators of a slot in one allocation: a solve at
// L = 14, D = 250 in 584 ms after 973, at L = 12, D = 200 in 347 after 552, setting up a site
// at L = 24, D = 1000 in 38.7 after 43. Loops of several callers run side by side; a caller works on
// its own loop, so it ends also when no worker is free. Without a holder every loop starts
// its own threads.
class Pool {
 public:
  struct Ref {
    Ref() { Pool::get().hold(1); }
    ~Ref() { Pool::get().hold(-1); }
    Ref(const Ref&) = delete;
    Ref& operator=(const Ref&) = delete;
  };
  struct Loop {
    void (*body)(void*, int tid);  // takes items until none is left; does not throw
    void* arg;
    int slots;                     // workers that may still join
    int tid = 1;                   // the next worker's number (the caller is 0)
    int active = 0;
  };
  static Pool& get() { return *instance(); }
  // Runs l.body on the caller and up to l.slots workers; false: no holder, nothing done.
  bool run(Loop& l) {
    {
      std::lock_guard<std::mutex> g(m_);
      if (holders_ == 0 || stop_) return false;
      try {
        while ((int)workers_.size() < std::min(l.slots, 63)) workers_.emplace_back([this] { work(); });
      } catch (const std::system_error&) {  // fewer threads, then
      }
      loops_.push_back(&l);
    }
    wake_.notify_all();
    l.body(l.arg, 0);
    std::unique_lock<std::mutex> g(m_);
    loops_.erase(std::remove(loops_.begin(), loops_.end(), &l), loops_.end());
    done_.wait(g, [&] { return l.active == 0; });
    return true;
  }

 private:
  // A forked child has none of the threads and none of their waits: it begins anew.
  static Pool*& instance() {
    static Pool* p = [] {
      pthread_atfork([] { get().m_.lock(); }, [] { get().m_.unlock(); },
                     [] {
                       const int holders = get().holders_;
                       instance() = new Pool;
                       get().holders_ = holders;
                     });
      return new Pool;  // its threads are gone once the last holder is
    }();
    return p;
  }
  void hold(int d) {
    std::vector<std::thread> gone;
    {
      std::unique_lock<std::mutex> g(m_);
      done_.wait(g, [&] { return !stop_; });  // another thread is taking the workers down
      holders_ += d;
      if (holders_ > 0 || workers_.empty()) return;
      stop_ = true;
      gone.swap(workers_);
    }
    wake_.notify_all();
    for (auto& t : gone) t.join();
    {
      std::lock_guard<std::mutex> g(m_);
      stop_ = false;
    }
    done_.notify_all();
  }
  void work() {
    std::unique_lock<std::mutex> g(m_);
    for (;;) {
      Loop* l = nullptr;
      wake_.wait(g, [&] {
        for (Loop* q : loops_)
          if (q->slots > 0) { l = q; return true; }
        return stop_;
      });
      if (!l) return;
      l->slots--;
      l->active++;
      const int tid = l->tid++;
      g.unlock();
      l->body(l->arg, tid);
      g.lock();
      l->slots = 0;  // no item is left: nobody else needs to join
      if (--l->active == 0) done_.notify_all();
    }
  }
  std::mutex m_;
  std::condition_variable wake_, done_;
  std::vector<Loop*> loops_;
  std::vector<std::thread> workers_;
  int holders_ = 0;
  bool stop_ = false;
};

// f(i, thread) for every i in [0, n), items handed out one at a time.
template <class F>
void parallel_for(int64_t n, int nthreads, F&& f) {
  nthreads = (int)std::max<int64_t>(1, std::min<int64_t>(nthreads, n));
  if (nthreads <= 1) {
    for (int64_t i = 0; i < n; i++) f(i, 0);
    return;
  }
  std::atomic<int64_t> next{0};
  std::exception_ptr err;
  std::mutex m;
  auto work = [&](int tid) {
    try {
      for (;;) {
        const int64_t i = next.fetch_add(1);
        if (i >= n) break;
        f(i, tid);
      }
    } catch (...) {
      std::lock_guard<std::mutex> g(m);
      if (!err) err = std::current_exception();
      next.store(n);
    }
  };
  using Work = decltype(work);
  Pool::Loop loop{[](void* w, int tid) { (*static_cast<Work*>(w))(tid); }, &work, nthreads - 1};
  if (!Pool::get().run(loop)) {
    std::vector<std::thread> pool;
    for (int t = 1; t < nthreads; t++) pool.emplace_back(work, t);
    work(0);
    for (auto& t : pool) t.join();
  }
  if (err) std::rethrow_exception(err);
}

}  // namespace chm
