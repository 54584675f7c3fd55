// Two helper threads for the copies between a caller's memory and pinned memory
// (uk_api.hip). One thread moves 33 to 42 GB/s of cold pages, less than the bus
// takes (50 each way); three together move 70 to 100.
//
// The crew is started by the first call that is large enough to use it and ends
// with the library. One call has it at a time, another that comes meanwhile does
// without. The helpers sleep between calls. While a call has them they poll for
// their next piece, 0.2 ms at most: waking takes 30 to 60 us, which is what a
// product between the copies often takes, and a longer one (or work that the
// caller's stream had before) costs no CPU time. A process with fewer than four
// CPUs has no crew.
#ifndef IREE_AMD_CSRC_HOST_CREW_H_
#define IREE_AMD_CSRC_HOST_CREW_H_

#include <pthread.h>
#include <signal.h>
#include <unistd.h>

#include <atomic>
#include <chrono>
#include <condition_variable>
#include <cstdint>
#include <mutex>
#include <system_error>
#include <thread>

namespace uk {

class HostCrew {
 public:
  static HostCrew& instance() {
    static Holder holder;
    return *holder.crew;
  }

  // Takes the crew for a call; false if another call has it or there are no threads to be had.
  bool engage() {
    if (!owner_.try_lock()) return false;
    if (!started_) {
      started_ = true;
      start();
    }
    if (!helpers_[0].joinable()) {
      owner_.unlock();
      return false;
    }
    {
      std::lock_guard<std::mutex> lock(mutex_);
      engaged_.store(true, std::memory_order_relaxed);
      ++engagements_;
      dozing_.store(0);
    }
    wake_.notify_all();
    return true;
  }
  void release() {
    engaged_.store(false, std::memory_order_relaxed);
    owner_.unlock();
  }

  // work(i) for every i < count, on the calling thread and whichever helpers are awake; i is handed out in ascending
  // order. `idle` is called now and then while the caller waits for the helpers' last pieces.
  template <typename Work, typename Idle>
  void run(uint32_t count, Work work, Idle idle) {
    call_ = [](void* w, uint32_t i) { (*(Work*)w)(i); };
    context_ = &work;
    count_ = count;
    next_.store(0, std::memory_order_relaxed);
    open_.store(true);
    // A helper that polled in vain says so before it looks for open work a last time: either it sees this work or it is
    // woken, once. (Not those that `engage` has just woken: a wake-up costs microseconds a time.)
    if (dozing_.load() != 0 && dozing_.exchange(0) != 0) {
      { std::lock_guard<std::mutex> lock(mutex_); }
      wake_.notify_all();
    }
    for (uint32_t i; (i = next_.fetch_add(1, std::memory_order_relaxed)) < count;) work(i);
    // A helper announces itself before it looks whether the work is still open: once none is announced after it has
    // been closed, none reads the fields above any more.
    open_.store(false);
    for (uint32_t spins = 1; active_.load() != 0; ++spins) {
      __builtin_ia32_pause();
      if (spins % (1u << 16) == 0) idle();
    }
  }

 private:
  // A forked child has no helpers to wait for: there the crew is left as it is.
  struct Holder {
    HostCrew* const crew = new HostCrew();
    const pid_t pid = getpid();
    ~Holder() {
      if (getpid() == pid) delete crew;
    }
  };

  HostCrew() {}
  ~HostCrew() {
    {
      std::lock_guard<std::mutex> lock(mutex_);
      stop_.store(true);
    }
    wake_.notify_all();
    for (std::thread& t : helpers_)
      if (t.joinable()) t.join();
  }

  void start() {
    if (std::thread::hardware_concurrency() < 4) return;
    sigset_t all, before;  // signals are for the program's own threads
    sigfillset(&all);
    pthread_sigmask(SIG_SETMASK, &all, &before);
    try {
      for (std::thread& t : helpers_) t = std::thread([this] { help(); });
    } catch (const std::system_error&) {
    }
    pthread_sigmask(SIG_SETMASK, &before, nullptr);
  }

  bool work_waits() const { return open_.load() && next_.load(std::memory_order_relaxed) < count_.load(std::memory_order_relaxed); }

  void help() {
    typedef std::chrono::steady_clock clock;
    constexpr std::chrono::microseconds kPolling(200);
    uint32_t seen = 0;  // engagements
    for (bool dozes = false;;) {
      {
        std::unique_lock<std::mutex> lock(mutex_);
        if (dozes) dozing_.fetch_add(1);
        wake_.wait(lock, [&] { return stop_.load() || engagements_ != seen || work_waits(); });
        if (stop_.load()) return;
        seen = engagements_;
      }
      dozes = false;
      clock::time_point idle_since = clock::now();
      for (uint32_t spins = 1; engaged_.load(std::memory_order_relaxed) && !stop_.load(std::memory_order_relaxed); ++spins) {
        if (work_waits()) {
          active_.fetch_add(1);
          if (open_.load()) {
            const uint32_t count = count_.load(std::memory_order_relaxed);
            for (uint32_t i; (i = next_.fetch_add(1, std::memory_order_relaxed)) < count;) call_(context_, i);
          }
          active_.fetch_sub(1);
          idle_since = clock::now();
        } else {
          __builtin_ia32_pause();
          if (spins % 64 == 0 && clock::now() - idle_since > kPolling) {
            dozes = true;
            break;
          }
        }
      }
    }
  }

  std::mutex owner_;
  bool started_ = false;
  std::thread helpers_[2];
  std::mutex mutex_;
  std::condition_variable wake_;
  uint32_t engagements_ = 0;  // (under mutex_)
  std::atomic<bool> stop_{false}, engaged_{false}, open_{false};
  std::atomic<uint32_t> next_{0}, active_{0}, count_{0}, dozing_{0};
  void (*call_)(void*, uint32_t) = nullptr;
  void* context_ = nullptr;
};

}  // namespace uk

#endif  // IREE_AMD_CSRC_HOST_CREW_H_
