// Host build of the wait for the host's copy of the counters
// (mcell_amd/csrc/poll.h) for tests/test_poll.py.
#include <stdint.h>

#include "../mcell_amd/csrc/poll.h"

extern "C" {

// A wait whose word comes at look `ready_at` (never: ~0) and whose stream is
// found at rest by the query number `rest_at` (never: ~0).  out: looks,
// pauses, yields, queries.
int poll(uint64_t ready_at, uint64_t rest_at, uint64_t* out) {
  uint64_t &looks = out[0], &pauses = out[1], &yields = out[2], &queries = out[3];
  looks = pauses = yields = queries = 0;
  return mcg::poll_until([&] { return looks++ >= ready_at; }, [&] { ++pauses; }, [&] { ++yields; },
                         [&] { return queries++ < rest_at; });
}

}  // extern "C"
