// Names the step a context's close is in when that step does not end. A close waits for things the library does not own
// (a copy engine, a stream of the engine, the HIP runtime's own teardown) and has no deadline: memory that a copy may
// still use cannot be given back. So a wait that lasts is reported, once per step, from a thread that makes no HIP call.
#pragma once

#include <chrono>
#include <condition_variable>
#include <cstdio>
#include <functional>
#include <mutex>
#include <thread>

namespace tsa {

class CloseWatch {
 public:
  using Report = std::function<void(const char* step, double seconds)>;
  explicit CloseWatch(std::chrono::milliseconds bound = std::chrono::seconds(10), Report report = to_stderr) noexcept
      : bound_(bound), report_(std::move(report)) {
    try {
      th_ = std::thread([this] { watch(); });
    } catch (...) {  // (no thread left: a close without a watch)
    }
  }
  ~CloseWatch() {
    {
      std::lock_guard<std::mutex> lk(mu_);
      step_ = nullptr;
      end_ = true;
    }
    cv_.notify_all();
    if (th_.joinable()) th_.join();
  }
  CloseWatch(const CloseWatch&) = delete;
  CloseWatch& operator=(const CloseWatch&) = delete;

  void step(const char* name) noexcept {  // name: a literal
    std::lock_guard<std::mutex> lk(mu_);
    step_ = name;
    since_ = Clock::now();
  }

 private:
  using Clock = std::chrono::steady_clock;
  static void to_stderr(const char* step, double seconds) {
    std::fprintf(stderr, "tierstream: ss_close is still waiting after %.0f s: %s\n", seconds, step);
  }
  void watch() {
    std::unique_lock<std::mutex> lk(mu_);
    Clock::time_point reported{};  // the start of the last step reported
    while (!end_) {
      const auto now = Clock::now();
      if (step_ && since_ != reported && now - since_ >= bound_) {
        reported = since_;
        report_(step_, std::chrono::duration<double>(now - since_).count());
      }
      // (a step is entered without waking this thread: it looks twice within a bound)
      cv_.wait_for(lk, bound_ / 2, [this] { return end_; });
    }
  }

  std::chrono::milliseconds bound_;
  Report report_;
  std::mutex mu_;
  std::condition_variable cv_;
  const char* step_ = nullptr;
  Clock::time_point since_{};
  bool end_ = false;
  std::thread th_;
};

}  // namespace tsa
