// A few threads of a context for work on host arrays that one thread's share of the memory bandwidth bounds.
#pragma once
#include <sched.h>
#include <unistd.h>

#include <condition_variable>
#include <functional>
#include <mutex>
#include <thread>
#include <vector>

namespace nnvhip {

// run(parts, f) calls f(0) .. f(parts - 1), each once, on the calling thread and the workers, and returns when all are done.
// f must not throw.  Workers start with the first call, no more than the process has CPUs beside the caller's (a host that gives
// none: the caller does all of it), and sleep in between.  One caller at a time, like the context it belongs to.
//
// A process that was forked off has no workers, only this object's memory, in whatever state the threads it does not have left
// it: it starts workers of its own where it needs them, and never touches the old ones' lock, conditions (destroying one waits
// for its waiters) and thread handles, which stay behind.
class HostPool {
 public:
  static constexpr int kWorkers = 3;  // at most
  HostPool() = default;
  HostPool(const HostPool&) = delete;
  HostPool& operator=(const HostPool&) = delete;
  ~HostPool() {
    if (own_ == nullptr || pid_ != getpid()) return;
    {
      std::lock_guard<std::mutex> lock(own_->mu);
      own_->stop = true;
    }
    own_->wake.notify_all();
    for (auto& t : own_->threads) t.join();
    delete own_;
  }
  void run(int parts, const std::function<void(int)>& f) {
    if (parts > 1 && (own_ == nullptr || pid_ != getpid())) start();
    if (parts < 2 || own_ == nullptr || own_->threads.empty()) {
      for (int i = 0; i < parts; ++i) f(i);
      return;
    }
    State& s = *own_;
    {
      std::lock_guard<std::mutex> lock(s.mu);
      s.f = &f;
      s.parts = parts;
      s.next = 0;
      s.left = parts;
    }
    s.wake.notify_all();
    std::unique_lock<std::mutex> lock(s.mu);
    s.work(lock);
    s.done.wait(lock, [&] { return s.left == 0; });
    s.f = nullptr;
  }

 private:
  struct State {
    std::mutex mu;
    std::condition_variable wake, done;
    std::vector<std::thread> threads;
    const std::function<void(int)>* f = nullptr;
    int parts = 0, next = 0, left = 0;
    bool stop = false;
    // Parts that nobody has taken yet; `lock` is held on entry and on return.
    void work(std::unique_lock<std::mutex>& lock) {
      while (next < parts) {
        const int i = next++;
        const std::function<void(int)>* g = f;
        lock.unlock();
        (*g)(i);
        lock.lock();
        if (--left == 0) done.notify_all();
      }
    }
  };
  void start() {
    own_ = nullptr;  // (a forked process: its parent's)
    pid_ = getpid();
    try {
      State* s = own_ = new State();
      cpu_set_t cpus;
      const int others = sched_getaffinity(0, sizeof cpus, &cpus) == 0 ? CPU_COUNT(&cpus) - 1 : kWorkers;
      s->threads.reserve(kWorkers);
      for (int i = 0; i < (others < kWorkers ? others : kWorkers); ++i)
        s->threads.emplace_back([s] {
          std::unique_lock<std::mutex> lock(s->mu);
          for (;;) {
            s->wake.wait(lock, [&] { return s->stop || s->next < s->parts; });
            if (s->stop) return;
            s->work(lock);
          }
        });
    } catch (const std::exception&) {  // (those that did start are enough)
    }
  }
  State* own_ = nullptr;
  pid_t pid_ = 0;  // the process that started them
};

}  // namespace nnvhip
