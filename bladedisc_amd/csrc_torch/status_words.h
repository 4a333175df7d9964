// Words of host memory that kernels answer through: a call borrows one, hands its address to a
// kernel and waits for the non-zero value that the kernel stores there, once.
#ifndef DQ8_STATUS_WORDS_H_
#define DQ8_STATUS_WORDS_H_

#include <atomic>
#include <chrono>
#include <cstdint>
#include <mutex>
#include <vector>

namespace dq8 {

class StatusWords {
 public:
  static constexpr int kStride = 32;   // a 128-byte line each
  // `page`: n * kStride words that stay allocated as long as any kernel may write them
  StatusWords(int32_t* page, int n) {
    for (int i = 0; i < n; ++i) free_.push_back(page + i * kStride);
  }
  // null when all are in use (then the caller takes one of its own)
  volatile int32_t* borrow() {
    std::lock_guard<std::mutex> guard(mu_);
    if (free_.empty()) return nullptr;
    volatile int32_t* w = free_.back();
    free_.pop_back();
    return w;
  }
  void give_back(volatile int32_t* w) {
    std::lock_guard<std::mutex> guard(mu_);
    free_.push_back(w);
  }

 private:
  std::mutex mu_;
  std::vector<volatile int32_t*> free_;
};

// A borrowed word.  It goes back to the pool only when no kernel can still write it: one whose
// answer is outstanding would tell its next borrower about another call's data.  `Own` is the
// memory of a word outside the pool (a tensor), allocated by `allocate` when the pool is empty.
template <typename Own>
class StatusWord {
 public:
  template <typename Allocate>
  StatusWord(StatusWords& pool, Allocate&& allocate) : pool_(pool), w_(pool.borrow()) {
    if (!w_) {
      own_ = new Own();
      try {
        w_ = allocate(own_);
      } catch (...) {
        delete own_;
        throw;
      }
    }
    *w_ = 0;
  }
  StatusWord(const StatusWord&) = delete;
  ~StatusWord() {
    if (outstanding_) return;            // dropped, its own memory as well
    if (own_) delete own_;
    else pool_.give_back(w_);
  }

  // The address for a kernel, which from here on owes an answer.
  int32_t* hand_out() {
    outstanding_ = true;
    return const_cast<int32_t*>(w_);
  }

  // Waits for the device's answer: reading the word costs a microsecond, a stream
  // synchronisation ten.  After a while (a long queue in front, or a stream that cannot answer,
  // such as one under capture) it is left to `synchronize`, which reports errors by throwing.
  template <typename Synchronize>
  int32_t wait(Synchronize&& synchronize) {
    const auto until = std::chrono::steady_clock::now() + std::chrono::milliseconds(5);
    for (int i = 0;; ++i) {
      const int32_t v = *w_;
      if (v != 0) {
        std::atomic_thread_fence(std::memory_order_acquire);
        outstanding_ = false;
        return v;
      }
      __builtin_ia32_pause();
      if ((i & 255) == 255 && std::chrono::steady_clock::now() > until) break;
    }
    settle(synchronize);
    return *w_;
  }

  // After a launch that failed part of the way: nothing is owed once the stream has drained.
  template <typename Synchronize>
  void settle(Synchronize&& synchronize) {
    synchronize();
    outstanding_ = false;
  }

 private:
  StatusWords& pool_;
  volatile int32_t* w_;
  Own* own_ = nullptr;
  bool outstanding_ = false;
};

}  // namespace dq8

#endif  // DQ8_STATUS_WORDS_H_
