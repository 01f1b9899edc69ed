// Host build of the launch sizes (mcell_amd/csrc/launch_sizes.h) for
// tests/test_launch_sizes.py.
#include "../mcell_amd/csrc/launch_sizes.h"

extern "C" {

uint32_t scatter(uint32_t molecules, uint32_t bins) { return mcg::scatter_workgroups(molecules, bins); }
uint32_t append(uint32_t entries) { return mcg::append_workgroups(entries); }

}  // extern "C"
