// gate.hpp -- how many threads are inside the engine, so that HIP graphs are recorded and replayed only while there is one.
//
// Contexts of their own may be used from several threads. With six threads at work (solves, batched PPR, sessions) one
// session's capture was reported invalid and the process aborted; no single thread has seen that, and which call of
// another thread does it is not shown. So a capture begins only if no other thread is inside a call of the engine, and
// calls that begin meanwhile wait for its end (a few milliseconds); with company, the launches are issued one by one,
// which gives the same results in the same time. Host code only.
#pragma once
#include <condition_variable>
#include <mutex>

namespace prhc {

class Gate {
 public:
  void enter() {
    std::unique_lock<std::mutex> lock(m_);
    ended_.wait(lock, [&] { return !capturing_; });
    ++calls_;
  }
  void leave() {
    std::lock_guard<std::mutex> lock(m_);
    --calls_;
  }
  // True if the caller, inside a call, is the only one; calls of other threads then wait until end_capture.
  bool begin_capture() {
    std::lock_guard<std::mutex> lock(m_);
    return capturing_ = calls_ == 1;
  }
  void end_capture() {
    {
      std::lock_guard<std::mutex> lock(m_);
      capturing_ = false;
    }
    ended_.notify_all();
  }
  bool alone() {
    std::lock_guard<std::mutex> lock(m_);
    return calls_ == 1;
  }

 private:
  std::mutex m_;
  std::condition_variable ended_;
  int calls_ = 0;
  bool capturing_ = false;
};

inline Gate &gate() {
  static Gate g;
  return g;
}

// Held by every call that may reach the device; calls within a call count once.
class Call {
 public:
  Call() {
    if (depth()++ == 0) gate().enter();
  }
  ~Call() {
    if (--depth() == 0) gate().leave();
  }
  Call(const Call &) = delete;
  Call &operator=(const Call &) = delete;

 private:
  static int &depth() {
    thread_local int d = 0;
    return d;
  }
};

}  // namespace prhc
