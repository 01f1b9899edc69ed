// Host build of the launch sizes (mcell_amd/csrc/launch_sizes.h) for
// tests/test_launch_sizes.py.
#include "../mcell_amd/csrc/launch_sizes.h"

extern "C" {

uint32_t scatter(uint32_t molecules, uint32_t bins) { return mcg::scatter_workgroups(molecules, bins); }
// Runs iterations of rounds through RoundSizes.  Round i is of phase
// rounds[6 i] and number rounds[6 i + 1] with the drain's form rounds[6 i +
// 2], moves rounds[6 i + 3] movers and brings rounds[6 i + 4] proposals and
// rounds[6 i + 5] deferred movers; out[2 i], out[2 i + 1]: what was expected.
void rounds(uint64_t n, const uint32_t* rounds, uint32_t* out) {
  mcg::RoundSizes s;
  for (uint64_t i = 0; i < n; ++i) {
    const uint32_t* r = rounds + 6 * i;
    out[2 * i] = s.expect_props(r[0], r[2], r[1], r[3]);
    out[2 * i + 1] = s.expect_deferred(r[0], r[2], r[1], r[3]);
    if (r[1] == 0) s.first_round(r[0], r[2], r[4], r[5]);
  }
}

uint32_t room(uint32_t expected, uint32_t bound) { return mcg::room_for(expected, bound); }

uint32_t append(uint32_t entries) { return mcg::append_workgroups(entries); }

}  // extern "C"
