// Waiting for a word that a kernel writes to host memory.
#pragma once

namespace mcg {

// Polls `ready` until it holds (returns true), or until `running` says that
// nothing more can come and `ready` still does not hold (false).  The wait is
// mostly tens of microseconds, so it starts by spinning (`pause` between two
// looks), some 30 us; from then on the thread gives its core away between two
// looks (`yield`), for the threads that drive other contexts: 100 iterations
// of 4,000 molecules each take eight contexts on one core 54 ms, and 117 by
// spinning alone (on two cores 47 and 65, on sixteen 45 and 46).  `running`
// (a call into the runtime) is asked seldom.
constexpr int kPollSpins = 1000;
constexpr int kPollsPerLook = 20000;

template <class Ready, class Pause, class Yield, class Running>
bool poll_until(Ready ready, Pause pause, Yield yield, Running running) {
  for (int k = 0;; ++k) {
    if (ready()) return true;
    if (k < kPollSpins) pause();
    else yield();
    if (k % kPollsPerLook == kPollsPerLook - 1 && !running()) return ready();
    if (k == kPollSpins + kPollsPerLook) k = kPollSpins;
  }
}

}  // namespace mcg
