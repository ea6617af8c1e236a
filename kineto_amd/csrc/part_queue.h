/*
 * part_queue.h — the parts of a document that have reached the host, for the threads that copy them on.
 * One thread sees parts arrive, in order; any thread takes the next one that is there.  Host code only.
 */
#ifndef KTJ_PART_QUEUE_H_
#define KTJ_PART_QUEUE_H_

#include <atomic>
#include <chrono>
#include <condition_variable>
#include <cstdint>
#include <mutex>
#include <thread>

namespace ktj {

/* A wait for something that is mostly there within microseconds: looked for without a break for much longer than a
 * part takes to cross (9 us) and the first one to arrive, then between naps, so that a wait that takes longer does
 * not keep a core.  (A nap of 20 us takes 70 or more.) */
class Patience {
 public:
  /* true: the wait has come to its naps */
  bool pause() {
    if (++looks_ < kLooks) {
      relax();
      return false;
    }
    std::this_thread::sleep_for(std::chrono::microseconds(20));
    return true;
  }
  static void relax() {
#if defined(__x86_64__)
    __builtin_ia32_pause();
#else
    std::this_thread::yield();
#endif
  }

 private:
  static constexpr unsigned kLooks = 12000; /* some 200 us */
  unsigned looks_ = 0;
};

/* A thread takes a part only once that is there: what has nothing to do sleeps, and as many threads are awake as
 * the parts keep busy.  With every part dealt out beforehand and each thread awake for its own, 1.03 GB into memory
 * that was there before (21.1 ms) took 125 ms of processor time, 59 MB (1.25 ms) 7.0 ms; now 86 ms and 4.5 ms in the
 * same time.  Sleeping after 400, 1500 or 6000 looks makes no difference to the sessions (medians of eight runs in
 * turn: 30 000 records 656, 663 and 662 us, 650 with all awake; 118 000 kernels 2783, 2772 and 2834, 2826 with all
 * awake), and 400 the most to the processor time. */
class PartQueue {
 public:
  explicit PartQueue(uint64_t n_parts) : n_(n_parts) {}
  PartQueue(const PartQueue&) = delete;
  PartQueue& operator=(const PartQueue&) = delete;

  /* the next part is there */
  void arrive() {
    arrived_.fetch_add(1);
    wake(false);
  }
  /* no further part will be: whoever waits goes */
  void give_up() {
    given_up_.store(true);
    wake(true);
  }
  bool try_take(uint64_t* part) {
    uint64_t k = next_.load();
    while (k < arrived_.load()) {
      if (!next_.compare_exchange_weak(k, k + 1)) continue;
      if (k + 1 == n_) wake(true);
      *part = k;
      return true;
    }
    return false;
  }
  /* for the thread that sees the parts arrive, which does better to look for the next one: a part that is there
   * while every other thread has one */
  bool try_help(uint64_t* part) { return waiting_.load() == 0 && try_take(part); }
  /* waits for a part; false: there will be none */
  bool take(uint64_t* part) {
    if (try_take(part)) return true;
    waiting_.fetch_add(1);
    const bool got = wait_and_take(part);
    waiting_.fetch_sub(1);
    return got;
  }

 private:
  static constexpr unsigned kLooks = 400; /* some 6 us */
  bool wait_and_take(uint64_t* part) {
    for (unsigned looks = 0;;) {
      if (try_take(part)) return true;
      if (over()) return false;
      if (++looks < kLooks) {
        Patience::relax();
        continue;
      }
      std::unique_lock<std::mutex> lock(mutex_);
      sleepers_.fetch_add(1); /* before the last look: whoever changes something after it sees a sleeper */
      while (next_.load() >= arrived_.load() && !over()) changed_.wait(lock);
      sleepers_.fetch_sub(1);
      looks = 0;
    }
  }
  bool over() const { return given_up_.load() || next_.load() >= n_; }
  void wake(bool all) {
    if (sleepers_.load() == 0) return;
    { std::lock_guard<std::mutex> lock(mutex_); } /* a sleeper that has just looked is waiting by now */
    if (all) changed_.notify_all();
    else changed_.notify_one();
  }

  const uint64_t n_;
  alignas(64) std::atomic<uint64_t> arrived_{0};
  alignas(64) std::atomic<uint64_t> next_{0};
  alignas(64) std::atomic<bool> given_up_{false};
  std::atomic<unsigned> waiting_{0}, sleepers_{0};
  std::mutex mutex_;
  std::condition_variable changed_;
};

}  // namespace ktj
#endif
