// Host build of the launch sizes (mcell_amd/csrc/launch_sizes.h) for
// tests/test_launch_sizes.py.
#include "../mcell_amd/csrc/launch_sizes.h"

extern "C" {

uint32_t scatter(uint32_t molecules, uint32_t bins) { return mcg::scatter_workgroups(molecules, bins); }

}  // extern "C"
