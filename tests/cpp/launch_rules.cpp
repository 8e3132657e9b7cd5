// The dispatch rules of csrc/launch_rules.h behind C functions, for tests/test_launch_rules.py.
#include "../../cuda-kernel-lab_amd/csrc/launch_rules.h"

extern "C" {
int rule_merge_ranges_sources(int ngroups, int B) { return pdattn::merge_ranges_sources(ngroups, B); }
}
