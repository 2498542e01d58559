// Host-only checks of csrc/gate.hpp: a capture begins only while its thread is the only one inside a call, and calls of
// other threads wait for its end.
#include <atomic>
#include <chrono>
#include <cstdio>
#include <thread>
#include <vector>

#include "gate.hpp"

using namespace prhc;

#define CHECK(x)                                          \
  do {                                                    \
    if (!(x)) {                                           \
      std::printf("line %d: %s\n", __LINE__, #x);         \
      return 1;                                           \
    }                                                     \
  } while (0)

int main() {
  CHECK(!gate().begin_capture());  // outside of any call
  {
    const Call outer;
    const Call inner;  // a call within a call counts once
    CHECK(gate().alone());
    CHECK(gate().begin_capture());
    gate().end_capture();
  }
  // Another thread inside a call: no capture, until it has left.
  std::atomic<int> step{0};
  std::thread other([&] {
    const Call call;
    step = 1;
    while (step != 2) std::this_thread::yield();
  });
  while (step != 1) std::this_thread::yield();
  bool refused;
  {
    const Call call;
    refused = !gate().begin_capture() && !gate().alone();
  }
  step = 2;
  other.join();
  CHECK(refused);
  // Calls that begin during a capture wait for its end.
  std::atomic<bool> capturing{false}, entered{false}, early{false};
  std::thread late;
  {
    const Call call;
    CHECK(gate().begin_capture());
    capturing = true;
    late = std::thread([&] {
      const Call c;
      entered = true;
      if (capturing) early = true;
    });
    std::this_thread::sleep_for(std::chrono::milliseconds(50));
    if (entered) early = true;
    capturing = false;
    gate().end_capture();
    while (!entered) std::this_thread::yield();
  }
  late.join();
  CHECK(!early);
  // Many threads: never a call beside a capture.
  std::atomic<int> inside{0}, bad{0}, captures{0};
  std::vector<std::thread> pool;
  for (int t = 0; t < 6; ++t)
    pool.emplace_back([&, t] {
      for (int i = 0; i < 3000; ++i) {
        const Call call;
        ++inside;
        if (i % 3 == t % 3 && gate().begin_capture()) {
          ++captures;
          for (int k = 0; k < 50; ++k)
            if (inside != 1) ++bad;
          gate().end_capture();
        }
        --inside;
        if (i % 64 == t) std::this_thread::yield();
      }
    });
  for (auto &t : pool) t.join();
  CHECK(bad == 0);
  std::printf("ok, %d captures\n", captures.load());
  return 0;
}
