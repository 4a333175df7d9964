// csrc_torch/status_words.h against kernels that answer in time, late and never; the "device" is
// this program.  Prints ok.
#include "status_words.h"

#include <cstdio>
#include <cstdlib>
#include <stdexcept>
#include <thread>

#define CHECK(c)                                              \
  do {                                                        \
    if (!(c)) {                                               \
      std::printf("%s:%d: %s\n", __FILE__, __LINE__, #c);    \
      std::exit(1);                                           \
    }                                                         \
  } while (0)

struct Own {
  static int alive;
  int32_t word = 0;
  Own() { ++alive; }
  ~Own() { --alive; }
};
int Own::alive = 0;

int main() {
  using Word = dq8::StatusWord<Own>;
  static int32_t page[2 * dq8::StatusWords::kStride];
  dq8::StatusWords pool(page, 2);
  auto allocate = [](Own* o) { return &o->word; };
  auto never = [] { std::printf("synchronised\n"), std::exit(1); };
  auto broken = [] { throw std::runtime_error("the stream failed"); };

  int32_t* first;
  {   // never handed out; then answered: back in the pool
    Word w(pool, allocate);
  }
  {
    Word w(pool, allocate);
    first = w.hand_out();
    std::thread device([&] { *(volatile int32_t*)first = 2; });
    CHECK(w.wait(never) == 2);
    device.join();
  }
  {   // an answer that only the synchronisation brings
    Word w(pool, allocate);
    int32_t* p = w.hand_out();
    CHECK(p == first && *p == 0);
    CHECK(w.wait([&] { *p = 1; }) == 1);
  }
  {   // a launch that failed, on a stream that drains: nothing is owed
    Word w(pool, allocate);
    CHECK(w.hand_out() == first);
    w.settle([] {});
  }
  int32_t* late;
  try {   // a wait that fails: the answer may still come, to nobody
    Word w(pool, allocate);
    late = w.hand_out();
    CHECK(late == first);
    w.wait(broken);
    CHECK(false);
  } catch (const std::runtime_error&) {
  }
  {
    Word w(pool, allocate);
    int32_t* p = w.hand_out();
    CHECK(p != late);
    *late = 2;                       // another call's answer
    CHECK(w.wait([&] { *p = 1; }) == 1);
  }
  {   // one word left: the second borrower has its own, freed unless an answer is outstanding
    Word a(pool, allocate);
    {
      Word b(pool, allocate);
      CHECK(Own::alive == 1 && b.hand_out() != late);
      b.settle([] {});
    }
    CHECK(Own::alive == 0);
    try {
      Word b(pool, allocate);
      b.hand_out();
      b.settle(broken);
    } catch (const std::runtime_error&) {
    }
    CHECK(Own::alive == 1);
  }
  std::printf("ok\n");
}
