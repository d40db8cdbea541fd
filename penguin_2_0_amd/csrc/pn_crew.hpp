// pn_crew.hpp -- a few host threads that split an index range with their caller, for the length
// of one library call (building a picture's records from staged fields).
#pragma once

#include <condition_variable>
#include <functional>
#include <mutex>
#include <system_error>
#include <thread>
#include <vector>

namespace pn {

// run(n, fn) calls fn(begin, end) over disjoint parts of [0, n) on every thread and returns when
// all are done.  Threads that cannot be started are done without; fn must not throw.
class Crew {
 public:
  explicit Crew(int nthreads) {
    threads_.reserve(nthreads > 1 ? nthreads - 1 : 0);
    for (int t = 1; t < nthreads; ++t) {
      try {
        threads_.emplace_back([this, t] { work(t); });
      } catch (const std::system_error&) {
        break;   // fewer threads; the caller's own share grows
      }
    }
  }
  Crew(const Crew&) = delete;
  Crew& operator=(const Crew&) = delete;
  ~Crew() {
    {
      std::lock_guard<std::mutex> l(m_);
      quit_ = true;
    }
    start_.notify_all();
    for (std::thread& t : threads_) t.join();
  }
  void run(long n, const std::function<void(long, long)>& fn) {
    const int k = static_cast<int>(threads_.size()) + 1;
    if (k > 1) {
      std::lock_guard<std::mutex> l(m_);
      n_ = n;
      fn_ = &fn;
      left_ = k - 1;
      ++round_;
    }
    if (k > 1) start_.notify_all();
    fn(0, n / k);   // the caller's part
    if (k > 1) {
      std::unique_lock<std::mutex> l(m_);
      done_.wait(l, [this] { return left_ == 0; });
    }
  }

 private:
  void work(int t) {
    long seen = 0;
    std::unique_lock<std::mutex> l(m_);
    for (;;) {
      start_.wait(l, [&] { return quit_ || round_ != seen; });
      if (quit_) return;
      seen = round_;
      const long n = n_, k = static_cast<long>(threads_.size()) + 1;
      const std::function<void(long, long)>* fn = fn_;
      l.unlock();
      (*fn)(n * t / k, n * (t + 1) / k);
      l.lock();
      if (--left_ == 0) done_.notify_one();
    }
  }
  std::vector<std::thread> threads_;
  std::mutex m_;
  std::condition_variable start_, done_;
  const std::function<void(long, long)>* fn_ = nullptr;
  long n_ = 0, round_ = 0;
  int left_ = 0;
  bool quit_ = false;
};

}  // namespace pn
