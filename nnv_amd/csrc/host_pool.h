// A few threads of a context for work on host arrays that one thread's share of the memory bandwidth bounds.
#pragma once
#include <condition_variable>
#include <functional>
#include <mutex>
#include <system_error>
#include <thread>
#include <vector>

namespace nnvhip {

// run(parts, f) calls f(0) .. f(parts - 1), each once, on the calling thread and the workers, and returns when all are done.
// f must not throw.  Workers start with the first call (a host that gives none: the caller does all of it) and sleep in
// between.  One caller at a time, like the context it belongs to.
class HostPool {
 public:
  static constexpr int kWorkers = 3;
  HostPool() = default;
  HostPool(const HostPool&) = delete;
  HostPool& operator=(const HostPool&) = delete;
  ~HostPool() {
    {
      std::lock_guard<std::mutex> lock(mu_);
      stop_ = true;
    }
    wake_.notify_all();
    for (auto& t : threads_) t.join();
  }
  void run(int parts, const std::function<void(int)>& f) {
    if (parts > 1 && !started_) start();
    if (parts < 2 || threads_.empty()) {
      for (int i = 0; i < parts; ++i) f(i);
      return;
    }
    {
      std::lock_guard<std::mutex> lock(mu_);
      f_ = &f;
      parts_ = parts;
      next_ = 0;
      left_ = parts;
    }
    wake_.notify_all();
    std::unique_lock<std::mutex> lock(mu_);
    work(lock);
    done_.wait(lock, [&] { return left_ == 0; });
    f_ = nullptr;
  }

 private:
  void start() {
    started_ = true;
    try {
      threads_.reserve(kWorkers);
      for (int i = 0; i < kWorkers; ++i)
        threads_.emplace_back([this] {
          std::unique_lock<std::mutex> lock(mu_);
          for (;;) {
            wake_.wait(lock, [&] { return stop_ || next_ < parts_; });
            if (stop_) return;
            work(lock);
          }
        });
    } catch (const std::exception&) {  // (those that did start are enough)
    }
  }
  // Parts that nobody has taken yet; `lock` is held on entry and on return.
  void work(std::unique_lock<std::mutex>& lock) {
    while (next_ < parts_) {
      const int i = next_++;
      const std::function<void(int)>* f = f_;
      lock.unlock();
      (*f)(i);
      lock.lock();
      if (--left_ == 0) done_.notify_all();
    }
  }
  std::mutex mu_;
  std::condition_variable wake_, done_;
  std::vector<std::thread> threads_;
  const std::function<void(int)>* f_ = nullptr;
  int parts_ = 0, next_ = 0, left_ = 0;
  bool stop_ = false, started_ = false;
};

}  // namespace nnvhip
