// fair_share.h -- shares of a fixed amount, given out in the order of asking.
#pragma once

#include <condition_variable>
#include <mutex>

namespace mm {

// What the holders have together.
struct ShareGate {
  std::mutex mu;
  std::condition_variable cv;
  long long used = 0;
  unsigned long long next = 0, turn = 0;  // tickets given out, ticket that is looked at
};

// `part` of `whole` for as long as it lives.  Waits until everyone who asked before
// has theirs and the part fits beside them, so that a large part is not passed over
// by small ones.
class FairShare {
 public:
  FairShare(ShareGate &g, long long part, long long whole) : g_(g), part_(part)
  {
    std::unique_lock<std::mutex> lk(g_.mu);
    const unsigned long long mine = g_.next++;
    g_.cv.wait(lk, [&] { return g_.turn == mine && g_.used + part_ <= whole; });
    g_.used += part_;
    g_.turn++;
    lk.unlock();
    g_.cv.notify_all();
  }
  ~FairShare()
  {
    {
      std::lock_guard<std::mutex> lk(g_.mu);
      g_.used -= part_;
    }
    g_.cv.notify_all();
  }
  FairShare(const FairShare &) = delete;
  FairShare &operator=(const FairShare &) = delete;

 private:
  ShareGate &g_;
  const long long part_;
};

}  // namespace mm
